// Plain FP64 recurrence with the vectors resident on the chip: one launch
// runs all M steps, where the per-step kernels of plain.hip take one launch
// each (2.7-3.0 us of kernel and about 1 us of gap for a model of any size up to
// some 100,000 states, far above its few KB to MB of traffic).
//
// A workgroup keeps x_n of its rows in LDS and each thread the rows' matrix
// entries, x_n and x_{n-1} in registers, so a step reads 2 H values per row from
// LDS (H: entries on either side of the diagonal), adds them in the reference's
// order with no fused multiply-add, writes one value back and passes one barrier.
// Nothing but moments goes to memory. What bounds it: LDS bandwidth (5 x 512 B
// per 64 rows and step for H = 2) above about 2000 rows, the barrier and one
// LDS round trip below. Measured per step, real H: 0.25 us at 600 states, 0.37
// at 1800, 0.65 at 4042 (per-step launches: 3.7-3.9 us with the gaps).
//
// Models beyond one workgroup (MULTI): the rows are cut into G chunks of C
// consecutive rows, one workgroup each, and a workgroup also computes a halo.
// With D = max |column - row| and k steps between exchanges, the halo of x_n
// is k D rows on either side; step s of a phase computes the rows within
// (k - 1 - s) D of the chunk, so after k steps the chunk is exact and the
// halo is taken from the two neighbours (C >= k D). The halo of x_{n-1} reaches
// (k - 1) D; its rows are published one step early. An exchange costs about
// 1.1 us of latency between two XCDs plus its bytes, hence several steps per
// exchange where D is small against C. 73,006 states (D = 422, C = 1024, k = 2):
// 1.31 us per step; 64,000 states (D = 64, C = 512, k = 8): 0.59 us.
//
// Waiting: the launch is cooperative, so all workgroups are resident, and every
// wait is bounded (one second, or another workgroup's give-up): the kernel
// then ends, and the caller runs the per-step kernels instead.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace tbtkx {
namespace {

// Complex value; unlike double2 the compiler keeps arrays of it in registers.
struct __attribute__((aligned(16))) Z2 {
	double x, y;
};

// FP64 arithmetic of one element as in plain.hip: no fused multiply-add.
// kStride: elements of an LDS vector, element 0 holding the constant 1, so that
// byte offsets fit 16 bits and both vectors fit the CU's 160 KB.
template <typename S> struct R64;
template <> struct R64<Z2> {
	__device__ static Z2 mul(Z2 a, Z2 c) {
#pragma clang fp contract(off)
		return Z2{a.x * c.x - a.y * c.y, a.x * c.y + a.y * c.x};
	}
	__device__ static Z2 add(Z2 a, Z2 b) {
#pragma clang fp contract(off)
		return Z2{a.x + b.x, a.y + b.y};
	}
	__device__ static Z2 neg(Z2 p) { return Z2{-p.x, -p.y}; }
	__device__ static Z2 pick(bool c, Z2 a, Z2 b) { return Z2{c ? a.x : b.x, c ? a.y : b.y}; }
	__device__ static Z2 num(double re) { return Z2{re, 0.0}; }
	__device__ static double part(Z2 a, int c) { return c ? a.y : a.x; }
	__device__ static Z2 make(double re, double im) { return Z2{re, im}; }
	__device__ static double2 moment(Z2 x) { return make_double2(x.x, x.y); }
	static constexpr int kStride = 4095;
};
template <> struct R64<double> {
	__device__ static double mul(double a, double c) {
#pragma clang fp contract(off)
		return a * c;
	}
	__device__ static double add(double a, double b) {
#pragma clang fp contract(off)
		return a + b;
	}
	__device__ static double neg(double p) { return -p; }
	__device__ static double pick(bool c, double a, double b) { return c ? a : b; }
	__device__ static double num(double re) { return re; }
	__device__ static double part(double a, int) { return a; }
	__device__ static double make(double re, double) { return re; }
	__device__ static double2 moment(double x) { return make_double2(x, 0.0); }
	static constexpr int kStride = 8190;
};

// Exchanged values travel as 16 bytes each: the low and the high word, each
// with a 32-bit tag beside it, so both 8-byte halves say by themselves that
// they have arrived. Stored and loaded at the device's coherence point (sc1);
// the loads are volatile, as they are polled.
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kCoherent = 16, kVolatile = (int)0x80000000;
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t b, uint32_t at, double v, uint32_t tag) {
	const u32x4 w = {(uint32_t)__double2loint(v), tag, (uint32_t)__double2hiint(v), tag};
	__builtin_amdgcn_raw_buffer_store_b128(w, b, at * 16u, 0, kCoherent | kVolatile);
}
__device__ __forceinline__ u32x4 get(__amdgpu_buffer_rsrc_t b, uint32_t at) {
	return __builtin_amdgcn_raw_buffer_load_b128(b, at * 16u, 0, kCoherent | kVolatile);
}

constexpr int16_t kSlotPad = -32768;
constexpr int kResThreads = 1024;
constexpr long long kWaitTicks = 100000000ll;   // of the 100 MHz clock: one second

template <typename S>
struct ResArgs {
	const int16_t *scol;
	const uint8_t *scode;          // palette codes, or null
	const S *sv1, *sv2;            // slot values of H/s and 2H/s (no palette)
	const S *pal, *diag;           // palette (256 + 256), diagonal (N + N)
	int N, W, C, D, k, G;
	const int64_t *from;           // per vector
	const int *toff;               // per vector: first entry of its to-list
	const int64_t *to;             // ascending per vector
	double2 *coef;
	int M;
	void *xg;                      // 16 bytes each: [parity][x, y][components][N]
	uint32_t xg_bytes;
	uint32_t epoch;
	uint32_t *err;
};

// A row's entries in CSR order: up to H before its (first) diagonal entry,
// the diagonal, up to H after it. Unused places hold the value -0.0 and the
// constant 1: adding their product -0.0 leaves every sum as it is (a complex
// zero may change its sign). R rows per thread; without MULTI workgroup b runs
// start vector b on the whole model.
template <typename S, int H, int R, bool MULTI>
__global__ __launch_bounds__(kResThreads) void resident_recurrence(ResArgs<S> a) {
#pragma clang fp contract(off)
	typedef R64<S> A;
	constexpr int T = kResThreads, kStride = A::kStride;
	__shared__ S buf[2 * kStride];
	__shared__ int stop;
	const int t = threadIdx.x;
	const int g = MULTI ? (int)blockIdx.x : 0;
	const int vec = MULTI ? 0 : (int)blockIdx.x;
	const int N = a.N, D = MULTI ? a.D : 0, k = MULTI ? a.k : 1;
	const int halo = k * D;
	const int r0 = MULTI ? g * a.C : 0;
	const int r1 = MULTI ? (r0 + a.C < N ? r0 + a.C : N) : N;
	const int w0 = MULTI ? (r0 > halo ? r0 - halo : 0) : 0;
	const int w1 = MULTI ? (r1 + halo < N ? r1 + halo : N) : N;
	const int win = w1 - w0, own = r1 - r0;
	// i-th row of the workgroup: its own rows first, then the halo in rings of
	// D rows, left and right; -1 outside the matrix.
	auto row_of = [&](int i) __attribute__((always_inline)) -> int {
		if (i < own) return r0 + i;
		if (!MULTI) return -1;
		const int d = i - own, q = d / (2 * D), o = d - q * 2 * D;
		if (q >= k) return -1;
		const int r = o < D ? r0 - (q + 1) * D + o : r1 + q * D + (o - D);
		return r < 0 || r >= N ? -1 : r;
	};
	// Byte offsets into a vector: pos of the row itself (0: no row), adr of
	// entry s (low half) and s + H (high half).
	S diag[R], val[R][2 * H], xo[R], yo[R];
	uint32_t adr[R][H], pos[R];
	bool hasd[R];
#pragma unroll
	for (int j = 0; j < R; j++) {
		const int r = row_of(t + T * j);
		pos[j] = r < 0 ? 0u : (uint32_t)(r - w0 + 1) * (uint32_t)sizeof(S);
	}
	auto row_at = [&](int j) __attribute__((always_inline)) {
		return (int)(pos[j] / (uint32_t)sizeof(S)) - 1 + w0;
	};
	auto at = [](const S *v, uint32_t o) __attribute__((always_inline)) -> const S & {
		return *reinterpret_cast<const S *>(reinterpret_cast<const char *>(v) + o);
	};
	auto load = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
		for (int j = 0; j < R; j++) {
#pragma unroll
			for (int s = 0; s < 2 * H; s++) val[j][s] = A::num(-0.0);
#pragma unroll
			for (int s = 0; s < H; s++) adr[j][s] = 0;
			diag[j] = A::num(-0.0);
			bool hd = false;
			const int r = row_at(j);
			int b = 0, c = H;
			for (int s = 0; s < a.W && pos[j]; s++) {
				const int64_t e = (int64_t)s * N + r;
				const int off = a.scol[e];
				if (off == kSlotPad) break;
				S v;
				if (a.scode) {
					const int q = a.scode[e];
					v = q == 255 ? a.diag[(first ? 0 : N) + r] : a.pal[(first ? 0 : 256) + q];
				} else {
					v = first ? a.sv1[e] : a.sv2[e];
				}
				if (off == 0 && !hd) {
					hd = true;
					diag[j] = v;
					continue;
				}
				int col = r + off - w0;
				if (col < 0 || col >= win) col = r - w0;
				const int u = hd ? c++ : b++;
				const uint32_t o = (uint32_t)(1 + col) * (uint32_t)sizeof(S);
#pragma unroll
				for (int z = 0; z < 2 * H; z++) {
					val[j][z] = A::pick(z == u, v, val[j][z]);
					adr[j][z % H] |= z == u ? (z < H ? o : o << 16) : 0u;
				}
			}
			hasd[j] = hd;
		}
	};
	load(true);
	if (t < 2) buf[t * kStride] = A::num(1.0);
	const int from = (int)a.from[vec];
	for (int i = t; i < win; i += T) buf[1 + i] = A::num(w0 + i == from ? 1.0 : 0.0);
#pragma unroll
	for (int j = 0; j < R; j++) {
		xo[j] = A::num(pos[j] != 0 && row_at(j) == from ? 1.0 : 0.0);
		yo[j] = A::num(0.0);
	}
	if (t == 0) stop = 0;
	// This workgroup's part of the to-list.
	int q0 = a.toff[vec], q1 = a.toff[vec + 1];
	if (MULTI) {
		int lo = q0, hi = q1;
		while (lo < hi) {
			const int m = (lo + hi) >> 1;
			if (a.to[m] < r0) lo = m + 1;
			else hi = m;
		}
		const int first = lo;
		hi = q1;
		while (lo < hi) {
			const int m = (lo + hi) >> 1;
			if (a.to[m] < r1) lo = m + 1;
			else hi = m;
		}
		q0 = first;
		q1 = lo;
	}
	const int my = q0 + t < q1 ? (int)a.to[q0 + t] - w0 + 1 : -1;
	__syncthreads();

	auto gather = [&](const S *cur, int n) __attribute__((always_inline)) {
		if (my >= 0) a.coef[(int64_t)(q0 + t) * a.M + n] = A::moment(cur[my]);
		for (int q = q0 + t + T; q < q1; q += T)
			a.coef[(int64_t)q * a.M + n] = A::moment(cur[(int)a.to[q] - w0 + 1]);
	};
	gather(buf, 0);

	// The first RN rows of every thread: x_n into dst from x_{n-1} in src.
	auto rows = [&](auto rn, auto first, const S *src, S *dst) __attribute__((always_inline)) {
		constexpr int RN = decltype(rn)::value;
		constexpr bool FIRST = decltype(first)::value;
#pragma unroll
		for (int j = 0; j < RN; j++) {
			S x[2 * H];
#pragma unroll
			for (int s = 0; s < H; s++) {
				x[s] = at(src, adr[j][s] & 0xffffu);
				x[s + H] = at(src, adr[j][s] >> 16);
			}
			S acc = FIRST ? A::num(0.0) : A::neg(yo[j]);
#pragma unroll
			for (int s = 0; s < H; s++) acc = A::add(acc, A::mul(val[j][s], x[s]));
			acc = A::add(acc, A::mul(diag[j], A::pick(hasd[j], xo[j], A::num(1.0))));
#pragma unroll
			for (int s = H; s < 2 * H; s++) acc = A::add(acc, A::mul(val[j][s], x[s]));
			yo[j] = xo[j];
			xo[j] = acc;
			if (pos[j]) const_cast<S &>(at(dst, pos[j])) = acc;
		}
	};
	auto step = [&](auto first, const S *src, S *dst, int need) __attribute__((always_inline)) {
		if constexpr (!MULTI) {
			rows(std::integral_constant<int, R>{}, first, src, dst);
		} else {
			const int rn = (need + T - 1) / T;
#define TBTKX_ROWS(Q)                                                                        \
	if constexpr (R >= Q)                                                                \
		if (rn == Q) rows(std::integral_constant<int, Q>{}, first, src, dst);
			TBTKX_ROWS(1)
			TBTKX_ROWS(2)
			TBTKX_ROWS(3)
			TBTKX_ROWS(4)
			TBTKX_ROWS(5)
			TBTKX_ROWS(6)
			TBTKX_ROWS(7)
			TBTKX_ROWS(8)
			TBTKX_ROWS(9)
			TBTKX_ROWS(10)
			TBTKX_ROWS(11)
			TBTKX_ROWS(12)
#undef TBTKX_ROWS
		}
		__syncthreads();
	};
	constexpr int NC = sizeof(S) / 8;
	const __amdgpu_buffer_rsrc_t xg =
	    __builtin_amdgcn_make_buffer_rsrc(a.xg, 0, MULTI ? a.xg_bytes : 0, 0x00027000);
	// Element of component c of vector v (0: x_n, 1: x_{n-1}) after phase p.
	auto slot_of = [&](int p, int v, int c, int r) __attribute__((always_inline)) {
		return (uint32_t)((((p & 1) * 2 + v) * NC + c) * N + r);
	};
	// Publish the current vector of the rows within `ext` of the chunk's
	// edges, as vector v of phase p.
	auto publish = [&](int p, int v, int ext) __attribute__((always_inline)) {
#pragma unroll
		for (int j = 0; j < R; j++) {
			const int i = t + T * j;
			if (i >= own) break;
			if ((g > 0 && i < ext) || (g < a.G - 1 && i >= own - ext)) {
#pragma unroll
				for (int c = 0; c < NC; c++)
					put(xg, slot_of(p, v, c, r0 + i), A::part(xo[j], c), a.epoch + (uint32_t)p);
			}
		}
	};
	// Take the neighbours' rows of phase p. Returns false when the wait was
	// given up.
	auto exchange = [&](S *cur, S *oth, int p) __attribute__((always_inline)) -> bool {
		const uint32_t want = a.epoch + (uint32_t)p;
		const long long begin = wall_clock64();
		// Per pass one row of the inner rings (x_n and x_{n-1}) and one of the
		// outermost ring (x_n only), all in flight together.
		const int inner = own + 2 * (k - 1) * D, outer = inner + 2 * D;
		int spins = 0;
		for (int i = t; own + i < inner || inner + i < outer; i += T) {
			const int ra = own + i < inner ? row_of(own + i) : -1;
			const int rb = inner + i < outer ? row_of(inner + i) : -1;
			u32x4 wa[2 * NC], wb[NC];
			const u32x4 none = {0, want, 0, want};
			for (;;) {
#pragma unroll
				for (int c = 0; c < NC; c++) {
					wb[c] = none;
					if (rb >= 0) wb[c] = get(xg, slot_of(p, 0, c, rb));
				}
#pragma unroll
				for (int c = 0; c < 2 * NC; c++) {
					wa[c] = none;
					if (ra >= 0) wa[c] = get(xg, slot_of(p, c / NC, c % NC, ra));
				}
				bool ok = true;
#pragma unroll
				for (int c = 0; c < NC; c++) ok = ok && wb[c].y == want && wb[c].w == want;
#pragma unroll
				for (int c = 0; c < 2 * NC; c++) ok = ok && wa[c].y == want && wa[c].w == want;
				if (ok) break;
				if ((++spins & 63) == 0 &&
				    (wall_clock64() - begin > kWaitTicks ||
				     __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
					__hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					stop = 1;
					break;
				}
			}
			auto value = [&](const u32x4 *w) __attribute__((always_inline)) {
				return A::make(__hiloint2double(w[0].z, w[0].x), __hiloint2double(w[NC - 1].z, w[NC - 1].x));
			};
			if (ra >= 0) {
				cur[1 + ra - w0] = value(wa);
				oth[1 + ra - w0] = value(wa + NC);
			}
			if (rb >= 0) cur[1 + rb - w0] = value(wb);
		}
		__syncthreads();
		if (stop) return false;
#pragma unroll
		for (int j = 0; j < R; j++) {
			if (t + T * j < own || !pos[j]) continue;
			xo[j] = at(cur, pos[j]);
			yo[j] = at(oth, pos[j]);
		}
		return true;
	};

	S *const xa = buf, *const xb = buf + kStride;
	int sub = 0, phase = 0, need = own + 2 * (k - 1) * D;
	auto after = [&](S *cur, S *oth, int n) __attribute__((always_inline)) -> bool {
		gather(cur, n);
		if (!MULTI) return true;
		need -= 2 * D;
		++sub;
		// x_{n-1} of the phase's end goes out one step ahead.
		if (sub == k - 1) publish(phase + 1, 1, halo - D);
		if (sub == k && n + 1 < a.M) {
			sub = 0;
			need = own + 2 * (k - 1) * D;
			publish(++phase, 0, halo);
			return exchange(cur, oth, phase);
		}
		return true;
	};
	if (a.M > 1) {
		step(std::true_type{}, xa, xb, need);
		load(false);
		if (!after(xb, xa, 1)) return;
	}
	int n = 2;
	for (; n + 1 < a.M; n += 2) {
		step(std::false_type{}, xb, xa, need);
		if (!after(xa, xb, n)) return;
		step(std::false_type{}, xa, xb, need);
		if (!after(xb, xa, n + 1)) return;
	}
	if (n < a.M) {
		step(std::false_type{}, xb, xa, need);
		after(xa, xb, n);
	}
}

__global__ __launch_bounds__(kThreads) void res_zero(uint32_t *p, int64_t n) {
	for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kThreads) p[i] = 0;
}

template <typename S, int H, int R, bool MULTI>
int launch_res(tbtkx_context *h, ResArgs<S> a, unsigned grid) {
	if constexpr (!MULTI) {
		resident_recurrence<S, H, R, MULTI><<<grid, kResThreads, 0, h->stream>>>(a);
		TBTKX_CHECK_HIP(hipGetLastError());
	} else {
		void *p[] = {&a};
		TBTKX_CHECK_HIP(hipLaunchCooperativeKernel(
		    (const void *)resident_recurrence<S, H, R, MULTI>, dim3(grid), dim3(kResThreads), p, 0,
		    h->stream));
	}
	return TBTKX_OK;
}

// Most rows per thread: what 128 VGPRs hold (16 wavefronts per CU) without
// scratch traffic that costs more than it saves; an entry takes 2.5 registers
// (complex 4.5), a row 7 more (11).
template <typename S, bool MULTI>
constexpr int max_rows(int H) {
	if (std::is_same<S, double>::value)
		return MULTI ? (H <= 1 ? 4 : H <= 3 ? 3 : 2) : (H <= 1 ? 8 : H == 2 ? 6 : H == 3 ? 4 : 3);
	return MULTI ? (H <= 2 ? 2 : 1) : (H <= 1 ? 4 : H == 2 ? 3 : 2);
}

template <typename S, int H, int R, bool MULTI>
int launch_res_r(tbtkx_context *h, const ResArgs<S> &a, unsigned grid, int r) {
	if constexpr (R <= max_rows<S, MULTI>(H)) {
		if (r <= R) return launch_res<S, H, R, MULTI>(h, a, grid);
		return launch_res_r<S, H, R + 1, MULTI>(h, a, grid, r);
	}
	set_error("resident recurrence: too many rows per thread");
	return TBTKX_ERR_STATE;
}

template <typename S, int H>
int launch_res_h(tbtkx_context *h, const ResArgs<S> &a, unsigned grid, int r) {
	return a.G > 1 ? launch_res_r<S, H, 1, true>(h, a, grid, r)
	               : launch_res_r<S, H, 1, false>(h, a, grid, r);
}

template <typename S>
int run_res(tbtkx_context *h, const ResidentPlan &plan, int V, const int64_t *from,
            const int *toff, const int64_t *to, int M) {
	const bool real = std::is_same<S, double>::value;
	const bool pal = h->use_palette && h->slot_pal;
	const size_t T = (size_t)toff[V];
	ResArgs<S> a{};
	a.scol = h->scol.as<int16_t>();
	a.scode = pal ? h->scode.as<uint8_t>() : nullptr;
	a.sv1 = real ? h->sv1r.as<S>() : h->sv1.as<S>();
	a.sv2 = real ? h->sv2r.as<S>() : h->sv2.as<S>();
	a.pal = real ? h->palr.as<S>() : h->pal.as<S>();
	a.diag = real ? h->pdiagr.as<S>() : h->pdiag.as<S>();
	a.N = (int)h->N;
	a.W = h->slot_W;
	a.D = (int)(h->band < h->N ? h->band : 0);
	a.k = plan.k;
	a.C = plan.C;
	a.G = (int)((h->N + plan.C - 1) / plan.C);
	a.M = M;
	int rc;
	// Start vectors, to-list and its offsets in one copy.
	std::vector<int64_t> &in = h->res_host;
	in.resize(V + T + (V + 2) / 2);
	memcpy(in.data(), from, (size_t)V * 8);
	memcpy(in.data() + V, to, T * 8);
	memcpy(in.data() + V + T, toff, (size_t)(V + 1) * 4);
	if ((rc = h->res_in.reserve(in.size() * 8))) return rc;
	if ((rc = h->coef.reserve((T > 0 ? T : 1) * M * 16))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->res_in.ptr, in.data(), in.size() * 8, hipMemcpyHostToDevice,
	                               h->stream));
	a.from = h->res_in.as<int64_t>();
	a.to = a.from + V;
	a.toff = reinterpret_cast<const int *>(a.from + V + T);
	a.coef = h->coef.as<double2>();
	if (a.G > 1) {
		// Tags are never used twice: a buffer starts all zero and the tags go on
		// from launch to launch.
		const size_t bytes = (size_t)h->N * sizeof(S) / 8 * 64;
		const uint32_t phases = (uint32_t)(M / plan.k + 2);
		if (!h->res_xg.ptr || h->res_xg.bytes < bytes || h->res_epoch > 0xffffffffu - phases) {
			if ((rc = h->res_xg.reserve(bytes))) return rc;
			if ((rc = h->res_err.reserve(256))) return rc;
			res_zero<<<1024, kThreads, 0, h->stream>>>(h->res_xg.as<uint32_t>(),
			                                           (int64_t)(h->res_xg.bytes / 4));
			res_zero<<<1, kThreads, 0, h->stream>>>(h->res_err.as<uint32_t>(), 64);
			h->res_epoch = 1;
		}
		a.xg = h->res_xg.ptr;
		a.xg_bytes = (uint32_t)bytes;
		a.err = h->res_err.as<uint32_t>();
		a.epoch = h->res_epoch;
		h->res_epoch += phases;
	}
	const int rows = a.G > 1 ? a.C + 2 * (a.k - 1) * a.D : a.N;
	const int r = (rows + kResThreads - 1) / kResThreads;
	const unsigned grid = a.G > 1 ? (unsigned)a.G : (unsigned)V;
	switch (h->slot_half) {
	case 0:
	case 1: return launch_res_h<S, 1>(h, a, grid, r);
	case 2: return launch_res_h<S, 2>(h, a, grid, r);
	case 3: return launch_res_h<S, 3>(h, a, grid, r);
	default: return launch_res_h<S, 4>(h, a, grid, r);
	}
}

}  // namespace

// The model fits one workgroup's registers and LDS, or chunks of it fit and
// their exchanges cost less than a launch per step. Times in us, from the
// measurements in this file's head; a launch per step takes 3.8 us up to
// 200,000 states and the slot step's bytes at 5.5 TB/s above.
ResidentPlan resident_plan(const tbtkx_context *h, int cus) {
	ResidentPlan best;
	const PlainForm f = plain_form(h);
	if (!h->use_resident || !f.slot || h->use_graph || h->slot_rows || h->use_patterns != 1 ||
	    h->slot_half > 4)
		return best;
	const bool real = h->real_path && h->h_real;
	const int H = h->slot_half;
	const int64_t N = h->N, D = h->band;
	const int window = (real ? R64<double>::kStride : R64<Z2>::kStride) - 1;
	const int one = real ? max_rows<double, false>(H) : max_rows<Z2, false>(H);
	const int many = real ? max_rows<double, true>(H) : max_rows<Z2, true>(H);
	// One round of rows (1024), and what a step takes without any.
	const double set = (real ? 0.025 : 0.06) * (2 * H + 1), base = 0.14;
	if (N <= (int64_t)one * kResThreads && N <= window) {
		best.C = (int)N;
		best.k = 1;
		best.us = base + set * (double)((N + kResThreads - 1) / kResThreads);
		return best;
	}
	if (D >= N) return best;
	double limit = std::max(3.8, f.bytes / 5.5e6);
	for (int k = 1; k <= 16; k++)
		for (int q = 1; q <= many; q++) {
			const int64_t C = (int64_t)q * kResThreads - 2 * (k - 1) * D;
			if (C < k * D || C + 2 * k * D > window || C >= N) continue;
			const int64_t G = (N + C - 1) / C;
			if (G > cus) continue;
			double us = 1.1 + (double)G * (2 * k - 1) * 2 * D * (real ? 32 : 64) / 8e6;
			for (int s = 0; s < k; s++)
				us += base + set * (double)((C + 2 * (k - 1 - s) * D + kResThreads - 1) / kResThreads);
			us /= k;
			if (us < limit) {
				limit = us;
				best.C = (int)C;
				best.k = k;
				best.us = us;
			}
		}
	return best;
}

int resident_moments(tbtkx_context *h, const ResidentPlan &plan, int V, const int64_t *from,
                     const int *toff, const int64_t *to, int M) {
	return h->real_path && h->h_real ? run_res<double>(h, plan, V, from, toff, to, M)
	                                 : run_res<Z2>(h, plan, V, from, toff, to, M);
}

int resident_given_up(tbtkx_context *h, const ResidentPlan &plan, bool *given_up) {
	*given_up = false;
	if (plan.C >= h->N) return TBTKX_OK;
	uint32_t err = 0;
	TBTKX_CHECK_HIP(hipMemcpyAsync(&err, h->res_err.ptr, 4, hipMemcpyDeviceToHost, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	if (err == 0) return TBTKX_OK;
	res_zero<<<1, kThreads, 0, h->stream>>>(h->res_err.as<uint32_t>(), 64);
	TBTKX_CHECK_HIP(hipGetLastError());
	*given_up = true;
	return TBTKX_OK;
}

}  // namespace tbtkx
