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
// Models beyond one workgroup (MULTI): the rows are seen as a grid of layers of L
// consecutive rows, and every column of the matrix lies `hq` layers and at
// most `ds` rows away from its row. The grid is cut into tiles of A layers x B
// rows, one workgroup each, and a workgroup also computes a halo. With k
// steps between exchanges the halo of x_n is k rings of hq layers and ds rows
// around the tile; step s of a phase computes the tile and k - 1 - s rings, so
// after k steps the tile is exact and the halo is taken from the neighbours
// (A >= k hq, B >= k ds). The halo of x_{n-1} has k - 1 rings; its rows are
// published one step early. L is a lattice's slowest stride (hq = 1), or the
// whole model (hq = 0: chunks of consecutive rows, ds = max |column - row|). A
// place of the window outside its layer is the row of that linear index, so
// bonds that wrap around within a layer need nothing special. An exchange costs
// about 1.3 us between two XCDs plus its bytes, hence several steps per exchange
// where the rings are small against the tile. Measured per step: 73,006 states
// (lattice 173 x 211 x 2) in 143 tiles of 16 x 33 rows, k = 4: 1.00 us; in chunks
// of 1024 consecutive rows (halo 422 rows a step), k = 2: 1.31 us.
//
// Waiting: the launch is cooperative, so all workgroups are resident, and every
// wait is bounded (one second, or another workgroup's give-up): the kernel
// then ends, and the caller runs the per-step kernels instead.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.hpp"
#include "tiles.hpp"

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
__device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t b, uint32_t at, double v, uint32_t tag) {
	const u32x4 w = {(uint32_t)__double2loint(v), tag, (uint32_t)__double2hiint(v), tag};
	__builtin_amdgcn_raw_buffer_store_b128(w, b, at * 16u, 0, kCoherent | kVolatile);
}
constexpr int16_t kSlotPad = -32768;
constexpr int kResThreads = 1024;

template <typename S>
struct ResArgs {
	const int16_t *scol;
	const uint8_t *scode;          // palette codes, or null
	const S *sv1, *sv2;            // slot values of H/s and 2H/s (no palette)
	const S *pal, *diag;           // palette (256 + 256), diagonal (N + N)
	int N, W, k, G;
	int L, La, hq, ds;             // rows per layer, layers, reach in layers and in rows
	int A, B, tb;                  // tile: layers, rows of each; tiles along a layer
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

// Entries q0 .. q1 - 1 of the ascending list `to` that lie in layers a .. a + h - 1
// of the tile's span of rows.
template <typename S>
__device__ __forceinline__ void span(const ResArgs<S> &a, const Tile &t, int *q0, int *q1) {
	const int64_t r0 = (int64_t)t.a * a.L + t.b, r1 = (int64_t)(t.a + t.h - 1) * a.L + t.b + t.w;
	auto first = [&](int64_t r) __attribute__((always_inline)) {
		int lo = *q0, hi = *q1;
		while (lo < hi) {
			const int m = (lo + hi) >> 1;
			if (a.to[m] < r) lo = m + 1;
			else hi = m;
		}
		return lo;
	};
	const int f = first(r0);
	*q1 = first(r1);
	*q0 = f;
}

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
	const int wave = __builtin_amdgcn_readfirstlane(t & ~63);   // its first thread
	const int g = MULTI ? (int)blockIdx.x : 0;
	const int vec = MULTI ? 0 : (int)blockIdx.x;
	const int N = a.N, k = MULTI ? a.k : 1, L = MULTI ? a.L : N;
	const int hq = MULTI ? a.hq : 0, ds = MULTI ? a.ds : 0;
	const Tile tile = MULTI ? tile_of(a.L, a.La, a.A, a.B, a.tb, g) : Tile{0, 0, 1, N};
	const Tile window = grown(tile, k * hq, k * ds);
	const int win = area(window), own = area(tile), P = window.w;
	// Rows within q rings of the tile.
	auto within = [&](int q) __attribute__((always_inline)) {
		return (tile.h + 2 * q * hq) * (tile.w + 2 * q * ds);
	};
	// Element of the window at a cell, and the row of an element (-1: none).
	auto place = [&](Cell c) __attribute__((always_inline)) {
		return (c.a - window.a) * P + c.b - window.b;
	};
	auto row_in = [&](int p) __attribute__((always_inline)) -> int {
		if (!MULTI) return p;
		const int q = p / P;
		const int64_t r = (int64_t)(window.a + q) * L + window.b + p - q * P;
		return r < 0 || r >= N ? -1 : (int)r;
	};
	// Element of the workgroup's i-th row: the tile, then the rings outwards;
	// -1: none.
	auto element = [&](int i) __attribute__((always_inline)) -> int {
		if (!MULTI) return i < own ? i : -1;
		if (i < own) return place(Cell{tile.a + i / tile.w, tile.b + i % tile.w});
		for (int q = 1; q <= k; q++)
			if (i < within(q))
				return place(frame_cell(grown(tile, q * hq, q * ds), i - within(q - 1), hq, ds));
		return -1;
	};
	// Byte offsets into a vector: pos of the row itself (0: no row), adr of
	// entry s (low half) and s + H (high half).
	S diag[R], val[R][2 * H], xo[R], yo[R];
	uint32_t adr[R][H], pos[R];
	bool hasd[R];
#pragma unroll
	for (int j = 0; j < R; j++) {
		const int p = element(t + T * j);
		pos[j] = p < 0 || row_in(p) < 0 ? 0u : (uint32_t)(p + 1) * (uint32_t)sizeof(S);
	}
	auto row_at = [&](int j) __attribute__((always_inline)) {
		return row_in((int)(pos[j] / (uint32_t)sizeof(S)) - 1);
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
				const int here = (int)(pos[j] / (uint32_t)sizeof(S)) - 1;
				const int lay = !MULTI || !hq ? 0 : 2 * off > L ? 1 : 2 * off < -L ? -1 : 0;
				int col = here + off - lay * (L - P);
				if (col < 0 || col >= win) col = here;
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
	for (int i = t; i < win; i += T) buf[1 + i] = A::num(row_in(i) == from ? 1.0 : 0.0);
#pragma unroll
	for (int j = 0; j < R; j++) {
		xo[j] = A::num(pos[j] != 0 && row_at(j) == from ? 1.0 : 0.0);
		yo[j] = A::num(0.0);
	}
	if (t == 0) stop = 0;
	// This workgroup's part of the to-list.
	int q0 = a.toff[vec], q1 = a.toff[vec + 1];
	if (MULTI) span(a, tile, &q0, &q1);
	// Element of the to-list's entry q, -1: of another tile.
	auto target = [&](int q) __attribute__((always_inline)) -> int {
		const int r = (int)a.to[q];
		if (!MULTI) return r;
		const int b = hq ? r % L : r;
		return b < tile.b || b >= tile.b + tile.w ? -1 : place(Cell{hq ? r / L : 0, b});
	};
	const int my = q0 + t < q1 ? target(q0 + t) : -1;
	__syncthreads();

	auto gather = [&](const S *cur, int n) __attribute__((always_inline)) {
		if (my >= 0) a.coef[(int64_t)(q0 + t) * a.M + n] = A::moment(cur[1 + my]);
		for (int q = q0 + t + T; q < q1; q += T) {
			const int p = target(q);
			if (p >= 0) a.coef[(int64_t)q * a.M + n] = A::moment(cur[1 + p]);
		}
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
			// Rounds with rows of this wavefront.
			const int rn = (need - wave + T - 1) / T;
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
	// Publish the current vector of the tile's rows within `ext` rings of its
	// edges, as vector v of phase p.
	auto publish = [&](int p, int v, int ext) __attribute__((always_inline)) {
#pragma unroll
		for (int j = 0; j < R; j++) {
			const int i = t + T * j;
			if (i >= own) break;
			const int la = i / tile.w, lb = i - la * tile.w;
			if (la < ext * hq || la >= tile.h - ext * hq || lb < ext * ds ||
			    lb >= tile.w - ext * ds) {
				const int r = (tile.a + la) * L + tile.b + lb;
#pragma unroll
				for (int c = 0; c < NC; c++)
					put(xg, slot_of(p, v, c, r), A::part(xo[j], c), a.epoch + (uint32_t)p);
			}
		}
	};
	// This thread's first rows of the inner rings and of the outermost.
	const int inner = within(k - 1), outer = within(k);
	int pa0 = -1, pb0 = -1, ra0 = -1, rb0 = -1;
	if (MULTI) {
		if (own + t < inner) pa0 = element(own + t);
		if (inner + t < outer) pb0 = element(inner + t);
		if (pa0 >= 0) ra0 = row_in(pa0);
		if (pb0 >= 0) rb0 = row_in(pb0);
	}
	// Take the neighbours' rows of phase p. Returns false when the wait was
	// given up.
	auto exchange = [&](S *cur, S *oth, int p) __attribute__((always_inline)) -> bool {
		const uint32_t want = a.epoch + (uint32_t)p;
		const long long begin = wall_clock64();
		// Per pass one row of the inner rings (x_n and x_{n-1}) and one of the
		// outermost ring (x_n only), all in flight together.
		int spins = 0;
		for (int i = t; own + i < inner || inner + i < outer; i += T) {
			int pa = pa0, pb = pb0, ra = ra0, rb = rb0;
			if (i != t) {
				pa = own + i < inner ? element(own + i) : -1;
				pb = inner + i < outer ? element(inner + i) : -1;
				ra = pa < 0 ? -1 : row_in(pa);
				rb = pb < 0 ? -1 : row_in(pb);
			}
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
				cur[1 + pa] = value(wa);
				oth[1 + pa] = value(wa + NC);
			}
			if (rb >= 0) cur[1 + pb] = value(wb);
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
	int sub = 0, phase = 0, need = inner;
	auto after = [&](S *cur, S *oth, int n) __attribute__((always_inline)) -> bool {
		gather(cur, n);
		if (!MULTI) return true;
		++sub;
		if (sub < k) need = within(k - 1 - sub);
		// x_{n-1} of the phase's end goes out one step ahead.
		if (sub == k - 1) publish(phase + 1, 1, k - 1);
		if (sub == k && n + 1 < a.M) {
			sub = 0;
			need = inner;
			publish(++phase, 0, k);
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

// Measured per step: 2,097,152 states (1024 x 1024 x 2) in 256 tiles of 64 x 128
// rows 2.7 us, where a launch per step took 11.9 (50 MB of vectors and 18 MB
// of matrix from the cache beyond L2); 1,048,576 states (512 x 512 x 4) 1.9 us;
// 864,000 states (96 x 100 x 90) 4.1 us, a frame of 2800 of 4000 rows there. Bound by
// VALU issue (62% of the SIMDs' cycles at 2,097,152 states: 8 FP64 and 12 integer
// instructions per row and step), the exchange, and LDS (busy 42% of the time).
// Large models (palette only): up to 8192 real rows per workgroup, one step per
// exchange. LDS holds one window of x_n, which is overwritten after a
// barrier; a row's entries are 16-bit window elements and 8-bit palette codes in
// registers, the palette's values come from LDS. The tile's frame comes first
// among its rows, so it is computed and published first and the exchange runs
// while the rest is computed. Element 0 of the window holds 1 and code 255 the
// value -0.0, for unused places.
constexpr int kWideBytes = 159200;
template <typename S, int H, int R>
__global__ __launch_bounds__(kResThreads) void resident_wide(ResArgs<S> a) {
#pragma clang fp contract(off)
	typedef R64<S> A;
	constexpr int T = kResThreads, NC = sizeof(S) / 8, CW = (2 * H + 3) / 4;
	__shared__ S buf[kWideBytes / sizeof(S)];
	__shared__ S pal[256];
	__shared__ int stop;
	const int t = threadIdx.x, N = a.N, L = a.L, hq = a.hq, ds = a.ds;
	const Tile tile = tile_of(a.L, a.La, a.A, a.B, a.tb, (int)blockIdx.x);
	const Tile window = grown(tile, hq, ds), inside = grown(tile, -hq, -ds);
	const int win = area(window), own = area(tile), P = window.w;
	const int frame = own - area(inside), ring = win - own;
	auto place = [&](Cell c) __attribute__((always_inline)) {
		return (c.a - window.a) * P + c.b - window.b;
	};
	auto row_in = [&](int p) __attribute__((always_inline)) -> int {
		const int q = p / P;
		const int64_t r = (int64_t)(window.a + q) * L + window.b + p - q * P;
		return r < 0 || r >= N ? -1 : (int)r;
	};
	S diag[R], xo[R], yo[R];
	uint32_t adr[R][H], code[R][CW], pos[R], hasd = 0;
#pragma unroll
	for (int j = 0; j < R; j++) {
		const int i = t + T * j;
		pos[j] = 0;
		if (i < frame) {
			pos[j] = place(frame_cell(tile, i, hq, ds)) + 1;
		} else if (i < own) {
			const int q = (i - frame) / inside.w;
			pos[j] = place(Cell{inside.a + q, inside.b + (i - frame) - q * inside.w}) + 1;
		}
	}
	auto diagonals = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
		for (int j = 0; j < R; j++) {
			diag[j] = A::num(-0.0);
			if (hasd >> j & 1) diag[j] = a.diag[(first ? 0 : N) + row_in((int)pos[j] - 1)];
		}
		if (t < 256) pal[t] = t == 255 ? A::num(-0.0) : a.pal[(first ? 0 : 256) + t];
	};
	const int from = (int)a.from[0];
#pragma unroll
	for (int j = 0; j < R; j++) {
#pragma unroll
		for (int s = 0; s < H; s++) adr[j][s] = 0;
#pragma unroll
		for (int s = 0; s < CW; s++) code[j][s] = 0xffffffffu;
		const int here = (int)pos[j] - 1, r = pos[j] ? row_in(here) : -1;
		bool hd = false;
		int b = 0, c = H;
		for (int s = 0; s < a.W && pos[j]; s++) {
			const int64_t e = (int64_t)s * N + r;
			const int off = a.scol[e];
			if (off == kSlotPad) break;
			const uint32_t q = a.scode[e];
			if (off == 0 && !hd) {
				hd = true;
				continue;
			}
			const int lay = !hq ? 0 : 2 * off > L ? 1 : 2 * off < -L ? -1 : 0;
			const uint32_t o = (uint32_t)(here + off - lay * (L - P) + 1);
			const int u = hd ? c++ : b++;
#pragma unroll
			for (int z = 0; z < 2 * H; z++) {
				adr[j][z % H] |= z == u ? (z < H ? o : o << 16) : 0u;
				code[j][z / 4] ^= z == u ? (q ^ 255u) << 8 * (z % 4) : 0u;
			}
		}
		hasd |= (uint32_t)hd << j;
		xo[j] = A::num(pos[j] != 0 && r == from ? 1.0 : 0.0);
		yo[j] = A::num(0.0);
	}
	diagonals(true);
	if (t == 0) {
		buf[0] = A::num(1.0);
		stop = 0;
	}
	for (int i = t; i < win; i += T) buf[1 + i] = A::num(row_in(i) == from ? 1.0 : 0.0);
	int q0 = a.toff[0], q1 = a.toff[1];
	span(a, tile, &q0, &q1);
	auto target = [&](int q) __attribute__((always_inline)) -> int {
		const int r = (int)a.to[q], b = hq ? r % L : r;
		return b < tile.b || b >= tile.b + tile.w ? -1 : place(Cell{hq ? r / L : 0, b});
	};
	const int my = q0 + t < q1 ? target(q0 + t) : -1;
	auto gather = [&](int n) __attribute__((always_inline)) {
		if (my >= 0) a.coef[(int64_t)(q0 + t) * a.M + n] = A::moment(buf[1 + my]);
		for (int q = q0 + t + T; q < q1; q += T) {
			const int p = target(q);
			if (p >= 0) a.coef[(int64_t)q * a.M + n] = A::moment(buf[1 + p]);
		}
	};
	const __amdgpu_buffer_rsrc_t xg = __builtin_amdgcn_make_buffer_rsrc(a.xg, 0, a.xg_bytes, 0x00027000);
	auto slot_of = [&](int n, int c, int r) __attribute__((always_inline)) {
		return (uint32_t)(((n & 1) * NC + c) * N + r);
	};
	const int r0 = t < frame ? row_in((int)pos[0] - 1) : -1;
	const int ph0 = t < ring ? place(frame_cell(window, t, hq, ds)) : -1;
	const int rh0 = ph0 < 0 ? -1 : row_in(ph0);
	// Waits for row r of x_n; false when the wait was given up.
	auto take = [&](int r, int n, S *x) __attribute__((always_inline)) {
		const uint32_t want = a.epoch + (uint32_t)n;
		const long long begin = wall_clock64();
		int spins = 0;
		for (;;) {
			u32x4 w[NC];
			bool ok = true;
#pragma unroll
			for (int c = 0; c < NC; c++) w[c] = get(xg, slot_of(n, c, r));
#pragma unroll
			for (int c = 0; c < NC; c++) ok = ok && w[c].y == want && w[c].w == want;
			if (ok) {
				*x = A::make(__hiloint2double(w[0].z, w[0].x),
				             __hiloint2double(w[NC - 1].z, w[NC - 1].x));
				return;
			}
			if ((++spins & 63) == 0 &&
			    (wall_clock64() - begin > kWaitTicks ||
			     __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
				__hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				stop = 1;
				return;
			}
		}
	};
	auto step = [&](auto first, int n) __attribute__((always_inline)) {
		constexpr bool FIRST = decltype(first)::value;
#pragma unroll
		for (int j = 0; j < R; j++) {
			S x[2 * H], v[2 * H];
			// The packed words stay packed: unpacked once for all steps, they would
			// take more registers than there are.
#pragma unroll
			for (int s = 0; s < H; s++) asm volatile("" : "+v"(adr[j][s]));
#pragma unroll
			for (int s = 0; s < CW; s++) asm volatile("" : "+v"(code[j][s]));
#pragma unroll
			for (int s = 0; s < H; s++) {
				x[s] = buf[adr[j][s] & 0xffffu];
				x[s + H] = buf[adr[j][s] >> 16];
			}
#pragma unroll
			for (int s = 0; s < 2 * H; s++) v[s] = pal[code[j][s / 4] >> 8 * (s % 4) & 255u];
			S acc = FIRST ? A::num(0.0) : A::neg(yo[j]);
#pragma unroll
			for (int s = 0; s < H; s++) acc = A::add(acc, A::mul(v[s], x[s]));
			acc = A::add(acc, A::mul(diag[j], A::pick(hasd >> j & 1, xo[j], A::num(1.0))));
#pragma unroll
			for (int s = H; s < 2 * H; s++) acc = A::add(acc, A::mul(v[s], x[s]));
			yo[j] = xo[j];
			xo[j] = acc;
			if (T * j < frame && t + T * j < frame) {
				const int r = j == 0 ? r0 : row_in((int)pos[j] - 1);
#pragma unroll
				for (int c = 0; c < NC; c++)
					put(xg, slot_of(n, c, r), A::part(acc, c), a.epoch + (uint32_t)n);
			}
		}
		const bool more = n + 1 < a.M;
		S h0 = A::num(0.0);
		if (more && rh0 >= 0) take(rh0, n, &h0);
		__syncthreads();
#pragma unroll
		for (int j = 0; j < R; j++)
			if (pos[j]) {
				asm volatile("" : "+v"(pos[j]));
				buf[pos[j]] = xo[j];
			}
		if (rh0 >= 0) buf[1 + ph0] = h0;
		for (int i = t + T; more && i < ring; i += T) {
			const int p = place(frame_cell(window, i, hq, ds)), r = row_in(p);
			if (r >= 0) take(r, n, &buf[1 + p]);
		}
		__syncthreads();
	};
	__syncthreads();
	gather(0);
	if (a.M > 1) {
		step(std::true_type{}, 1);
		if (stop) return;
		gather(1);
		diagonals(false);
		__syncthreads();
	}
	for (int n = 2; n < a.M; n++) {
		step(std::false_type{}, n);
		if (stop) return;
		gather(n);
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
		return TBTKX_OK;
	} else {
		void *p[] = {&a};
		return launch_cooperative(h, (const void *)resident_recurrence<S, H, R, MULTI>, grid,
		                          kResThreads, p);
	}
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

// The same of the wide kernel: a row takes 3 values, H + (2 H + 3) / 4 words and
// its element.
template <typename S>
constexpr int wide_rows(int H) {
	if (std::is_same<S, double>::value) return H <= 2 ? 8 : H == 3 ? 7 : 5;
	return H <= 2 ? 4 : H == 3 ? 3 : 2;
}

template <typename S, int H, int R>
int launch_wide(tbtkx_context *h, ResArgs<S> a, unsigned grid, int r) {
	if constexpr (R <= wide_rows<S>(H)) {
		if (r > R) return launch_wide<S, H, R + 1>(h, a, grid, r);
		void *p[] = {&a};
		return launch_cooperative(h, (const void *)resident_wide<S, H, R>, grid, kResThreads, p);
	}
	set_error("resident recurrence: too many rows per thread");
	return TBTKX_ERR_STATE;
}

template <typename S, int H>
int launch_res_h(tbtkx_context *h, const ResArgs<S> &a, unsigned grid, int r, bool wide) {
	if (wide) return launch_wide<S, H, 1>(h, a, grid, r);
	return a.G > 1 ? launch_res_r<S, H, 1, true>(h, a, grid, r)
	               : launch_res_r<S, H, 1, false>(h, a, grid, r);
}

}  // namespace

// Tags are never used twice: a buffer starts all zero and the tags go on from
// launch to launch.
int exchange_buffer(tbtkx_context *h, size_t bytes, uint32_t phases) {
	if (h->res_err.ptr && (bytes == 0 || (h->res_xg.ptr && h->res_xg.bytes >= bytes)) &&
	    h->res_epoch <= 0xffffffffu - phases)
		return TBTKX_OK;
	int rc;
	if ((rc = h->res_xg.reserve(std::max<size_t>(bytes, 64))) || (rc = h->res_err.reserve(256))) {
		(void)hipGetLastError();
		return rc == TBTKX_ERR_OOM ? kDeclined : rc;
	}
	res_zero<<<1024, kThreads, 0, h->stream>>>(h->res_xg.as<uint32_t>(), (int64_t)(h->res_xg.bytes / 4));
	res_zero<<<1, kThreads, 0, h->stream>>>(h->res_err.as<uint32_t>(), 64);
	TBTKX_CHECK_HIP(hipGetLastError());
	h->res_epoch = 1;
	return TBTKX_OK;
}

namespace {

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
	a.k = plan.k;
	a.G = plan.G;
	a.L = plan.L;
	a.La = (int)(h->N / plan.L);
	a.hq = plan.hq;
	a.ds = plan.ds;
	a.A = plan.A;
	a.B = plan.B;
	a.tb = (plan.L + plan.B - 1) / plan.B;
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
		const size_t bytes = (size_t)h->N * sizeof(S) / 8 * (plan.wide ? 32 : 64);
		const uint32_t phases = (uint32_t)(M / plan.k + 2);
		if ((rc = exchange_buffer(h, bytes, phases))) return rc;
		a.xg = h->res_xg.ptr;
		a.xg_bytes = (uint32_t)bytes;
		a.err = h->res_err.as<uint32_t>();
		a.epoch = h->res_epoch;
		h->res_epoch += phases;
	}
	const int q = 2 * (a.k - 1);
	const int rows = a.G > 1 ? (a.A + q * a.hq) * (a.B + q * a.ds) : a.N;
	const int r = (rows + kResThreads - 1) / kResThreads;
	const unsigned grid = a.G > 1 ? (unsigned)a.G : (unsigned)V;
	switch (h->slot_half) {
	case 0:
	case 1: return launch_res_h<S, 1>(h, a, grid, r, plan.wide);
	case 2: return launch_res_h<S, 2>(h, a, grid, r, plan.wide);
	case 3: return launch_res_h<S, 3>(h, a, grid, r, plan.wide);
	default: return launch_res_h<S, 4>(h, a, grid, r, plan.wide);
	}
}

}  // namespace

int64_t one_workgroup_rows(const tbtkx_context *h) {
	const bool real = h->real_path && h->h_real;
	const int H = h->slot_half;
	if (H > 4) return 0;
	const int64_t rows = (int64_t)kResThreads * (real ? max_rows<double, false>(H) : max_rows<Z2, false>(H));
	return std::min<int64_t>(rows, (real ? R64<double>::kStride : R64<Z2>::kStride) - 1);
}

// The model fits one workgroup's registers and LDS, or tiles of it fit and
// their exchanges cost less than a launch per step. Times in us, fitted to
// (model and measured, real H, H = 2 unless said): narrow, 73,006 states k = 1 1.9
// 1.8, k = 2 1.3 1.4, k = 4 1.0 1.0, k = 8 1.1 1.1; 524,288 states k = 4 1.6 1.8;
// wide, 73,006 states 1.6 1.6, 524,288 states 2.0 2.1, 2,097,152 states 3.0 2.7,
// 1,048,576 states H = 3 2.8 1.9, 864,000 states H = 3 4.6 4.1. A launch per step
// takes 2.7 us up to 200,000 states and the slot step's bytes at 5.5 TB/s above.
static ResidentPlan make_plan(const tbtkx_context *h, const PlainForm &f, int cus) {
	ResidentPlan best;
	if (!h->use_resident || !f.slot || h->use_graph || h->slot_rows || h->use_patterns != 1 ||
	    h->slot_half > 4)
		return best;
	const bool real = h->real_path && h->h_real;
	const int H = h->slot_half;
	const int64_t N = h->N, T = kResThreads;
	const int64_t window = (real ? R64<double>::kStride : R64<Z2>::kStride) - 1;
	const int64_t wide_window = kWideBytes / (real ? 8 : 16) - 1;
	const int many = real ? max_rows<double, true>(H) : max_rows<Z2, true>(H);
	const int wide = !f.pal ? 0 : real ? wide_rows<double>(H) : wide_rows<Z2>(H);
	// One round of rows (1024), and what a step takes without any.
	const double set = (real ? 0.025 : 0.06) * (2 * H + 1), base = 0.14;
	if (N <= one_workgroup_rows(h)) {
		best.C = best.L = best.B = (int)N;
		best.A = 1;
		best.us = base + set * (double)((N + T - 1) / T);
		return best;
	}
	if (!cooperative_now(h)) return best;
	double limit = std::max(2.7, f.bytes / 5.5e6);
	// Tiles of every form that fits and has no more of them than CUs.
	auto tiles = [&](int64_t L, int64_t hq, int64_t ds) {
		const int64_t La = N / L;
		if (ds <= 0 || (int64_t)cus * T * std::max(many, wide) < N) return;
		for (int64_t ta = 1; ta <= (hq ? std::min<int64_t>(La, cus) : 1); ta++) {
			const int64_t A = (La + ta - 1) / ta, tb0 = cus / ta;
			if ((La + A - 1) / A != ta) continue;
			// As few tiles along a layer as fit cost no more than twice the rows.
			for (int64_t tb = std::max<int64_t>(1, tb0 / 2); tb <= tb0; tb++) {
				const int64_t B = (L + tb - 1) / tb;
				if ((L + B - 1) / B != tb || ta * tb < 2) continue;
				const int64_t low = std::min(La - (ta - 1) * A, A), narrow = L - (tb - 1) * B;
				double steps = 0;                     // of a phase, without the exchange
				for (int64_t k = 0; k <= 16; k++) {   // 0: the wide kernel
					const int64_t q = k ? k : 1;
					if (low < q * hq || narrow < q * ds) break;
					if (k == 0 && (low < 2 * hq || narrow < 2 * ds)) continue;
					auto rows = [&](int64_t i) { return (A + 2 * i * hq) * (B + 2 * i * ds); };
					if (rows(q) > (k ? window : wide_window)) break;
					if (rows(q - 1) > T * (k ? many : wide)) {
						if (k) break;
						continue;
					}
					const double bytes = (double)(ta * tb) * (real ? 32 : 64) *
					                     ((double)(rows(q) - rows(0)) + (double)(rows(q - 1) - rows(0)));
					double us;
					if (k) {
						const int64_t most = std::max(rows(q) - rows(q - 1), rows(q - 1) - rows(0));
						steps += 0.5 + set * (double)rows(q - 1) / T;
						us = (1.3 * (double)((most + T - 1) / T) + bytes / 8e6 + steps) / (double)k;
					} else {
						us = 1.5 + bytes / 8e6 + set * (double)((rows(0) + T - 1) / T);
					}
					if (us < limit) {
						limit = us;
						best.C = (int)std::min<int64_t>(A * B, N - 1);
						best.k = (int)q;
						best.G = (int)(ta * tb);
						best.L = (int)L;
						best.hq = (int)hq;
						best.ds = (int)ds;
						best.A = (int)A;
						best.B = (int)B;
						best.wide = k == 0;
						best.us = us;
					}
				}
			}
		}
	};
	if (h->tile_L) tiles(h->tile_L, 1, h->tile_ds);
	if (h->band < N) tiles(N, 0, h->band);
	return best;
}

// The plan is made once per model and form.
ResidentPlan resident_plan(tbtkx_context *h, int cus) {
	const PlainForm f = plain_form(h);
	const int64_t key[8] = {h->csr_gen, h->N, h->Z, h->slot_half + 16 * (int64_t)h->tile_L, h->band,
	                        f.slot + 2 * f.pal + 4 * (h->real_path && h->h_real),
	                        (int64_t)h->use_resident + 2 * h->use_graph + 4 * h->slot_rows +
	                            64 * h->use_patterns,
	                        cus * 2 + cooperative_now(h)};
	if (memcmp(key, h->res_plan_key, sizeof key) != 0) {
		h->res_plan = make_plan(h, f, cus);
		memcpy(h->res_plan_key, key, sizeof key);
	}
	return h->res_plan;
}

int resident_moments(tbtkx_context *h, const ResidentPlan &plan, int V, const int64_t *from,
                     const int *toff, const int64_t *to, int M) {
	return h->real_path && h->h_real ? run_res<double>(h, plan, V, from, toff, to, M)
	                                 : run_res<Z2>(h, plan, V, from, toff, to, M);
}

int exchange_given_up(tbtkx_context *h, bool *given_up) {
	*given_up = false;
	uint32_t err = 0;
	TBTKX_CHECK_HIP(hipMemcpyAsync(&err, h->res_err.ptr, 4, hipMemcpyDeviceToHost, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	if (err == 0) return TBTKX_OK;
	res_zero<<<1, kThreads, 0, h->stream>>>(h->res_err.as<uint32_t>(), 64);
	TBTKX_CHECK_HIP(hipGetLastError());
	*given_up = true;
	return TBTKX_OK;
}

int resident_given_up(tbtkx_context *h, const ResidentPlan &plan, bool *given_up) {
	*given_up = false;
	return plan.G > 1 ? exchange_given_up(h, given_up) : TBTKX_OK;
}

}  // namespace tbtkx
