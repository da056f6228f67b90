// FP32 blocks of a real H with the vectors resident on the chip: one launch runs
// all steps of as many columns as fit, where the step kernels of block.hip and
// multi.hip stream every Phi_n through memory once per step (12 bytes per
// column element and step, at 4.4 TB/s).
//
// Columns are independent, so the chip is split into teams that take 8 columns
// each; a team's workgroups take a tile of the rows each (tiles.hpp) and
// exchange a halo of one ring after every step. Phi_n of the tile and its halo
// lie in LDS (two planes of 4 columns, so that neighbouring rows' 16-byte reads
// spread over all banks), Phi_{n-1} in registers; a row's entries are window
// elements and palette codes in registers. The tile's frame comes first among its
// rows and is published at once, so the exchange runs beside the rest. Values
// are stored as FP32, rows summed in FP64 and rounded once, dots summed in FP64,
// as in the step kernels.
//
// 512 threads with 256 registers each: 8 rows of 8 columns take 64 registers of
// Phi_{n-1} and 64 of entries; the dots are summed while the window is written,
// where no row's sums take registers. Bound by VALU issue (51% of the SIMDs' cycles on
// the first model below, 37% of it conversions between FP32 and FP64) at two
// wavefronts per SIMD that wait half of the time, and by the exchange; LDS is busy 23%
// of the time (32 bytes per entry, row and step). Two workgroups of 4 columns per CU
// spilled at 8 rows (46 us for 16 columns of the first model below against 24).
// A model too large for one pass takes several launches, 8 columns per team each.
//
// Measured per step, the step kernels and this one (dots):
// 1,048,576 states (512 x 512 x 4), 256 columns: 711, 356 us
// 159,520 states (40 x 997 x 4), 37 columns, gathered: 20.4, 7.8 us
//
// Waiting is bounded as in resident.hip; after a give-up the caller runs the
// step kernels.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "common.hpp"
#include "tiles.hpp"

namespace tbtkx {
namespace {

constexpr int kT = 512, kCols = 8, kDots = 20;
constexpr int kWin = 4956;        // window rows: 2 planes of 16 bytes a row in LDS
constexpr int kMaxRows = 8;       // per thread
constexpr uint64_t kEmpty = 0x7ff8a5a5c3c3e1e1ull;

// One model's scan: hash table of its distinct off-diagonal values of 2H/s (slot
// index = palette code), column offsets seen (offset + 32768), most entries
// beside slot 0, and whether something does not fit.
struct Scan {
	uint64_t key[256];
	uint32_t seen[2048];
	uint32_t ne, bad, pad[2];
};
struct ScanModel {
	int64_t N, e0;
	int W, pad;
};

__device__ __forceinline__ uint32_t hash8(uint64_t k) { return (uint32_t)((k * 0x9E3779B97F4A7C15ull) >> 56); }
// Inserts k into a table of 256; false when it is full.
__device__ __forceinline__ bool insert(uint64_t *table, uint64_t k) {
	uint32_t s = hash8(k);
	for (int i = 0; i < 256; i++, s = (s + 1) & 255u) {
		if (*(volatile uint64_t *)&table[s] == k) return true;
		const uint64_t was = atomicCAS((unsigned long long *)&table[s], (unsigned long long)kEmpty,
		                               (unsigned long long)k);
		if (was == kEmpty || was == k) return true;
	}
	return false;
}

__global__ __launch_bounds__(kThreads) void scan_init(Scan *s) {
	Scan &d = s[blockIdx.x];
	for (int i = threadIdx.x; i < 256; i += kThreads) d.key[i] = kEmpty;
	for (int i = threadIdx.x; i < 2048; i += kThreads) d.seen[i] = 0;
	if (threadIdx.x == 0) d.ne = d.bad = 0;
}

__global__ __launch_bounds__(kThreads) void scan_model(const ScanModel *__restrict__ models,
                                                       const uint32_t *__restrict__ ecol,
                                                       const double *__restrict__ ev2, Scan *out) {
	__shared__ unsigned long long key[256];
	__shared__ uint32_t seen[2048], ne, bad;
	const ScanModel m = models[blockIdx.y];
	for (int i = threadIdx.x; i < 256; i += kThreads) key[i] = kEmpty;
	for (int i = threadIdx.x; i < 2048; i += kThreads) seen[i] = 0;
	if (threadIdx.x == 0) ne = bad = 0;
	__syncthreads();
	uint32_t most = 0, wrong = 0;
	for (int64_t r = (int64_t)blockIdx.x * kThreads + threadIdx.x; r < m.N;
	     r += (int64_t)gridDim.x * kThreads) {
		for (int u = 0; u < m.W; u++) {
			const int64_t e = m.e0 + r * m.W + u;
			const uint64_t k = (uint64_t)__double_as_longlong(ev2[e]);
			const int64_t off = (int64_t)ecol[e] - r;
			if (u == 0) {
				wrong |= off != 0;
				continue;
			}
			if (off < -32767 || off > 32767 || k == kEmpty) {
				wrong = 1;
				continue;
			}
			if (off != 0 || (k << 1) != 0) most = u > (int)most ? (uint32_t)u : most;
			if (off != 0) {
				const uint32_t o = (uint32_t)(off + 32768), bit = 1u << (o & 31);
				if (!(*(volatile uint32_t *)&seen[o >> 5] & bit)) atomicOr(&seen[o >> 5], bit);
			}
			if (!insert((uint64_t *)key, k)) wrong = 1;
		}
	}
	if (most) atomicMax(&ne, most);
	if (wrong) bad = 1;
	__syncthreads();
	Scan &d = out[blockIdx.y];
	for (int i = threadIdx.x; i < 256; i += kThreads)
		if (key[i] != kEmpty && !insert(d.key, key[i])) bad = 1;
	for (int i = threadIdx.x; i < 2048; i += kThreads)
		if (seen[i]) atomicOr(&d.seen[i], seen[i]);
	__syncthreads();
	if (threadIdx.x == 0) {
		atomicMax(&d.ne, ne);
		if (bad) atomicOr(&d.bad, 1u);
	}
}

// Sums K values over the wavefront (K = 16 or 4): the two swaps halve the values
// a lane holds, rotations within 16 lanes do the rest. Value i + K/2 (r / 2) + K/4 (r
// % 2), i < K/4, ends in v[i] of the lanes of row r (16 lanes). Through ds_bpermute
// the 20 sums took 4 us of a step.
template <int K>
__device__ __forceinline__ void wave_sums(double *v) {
	auto halves = [&](auto swap, int n) __attribute__((always_inline)) {
#pragma unroll
		for (int i = 0; i < n; i++) {
			const auto lo = swap((uint32_t)__double2loint(v[i]), (uint32_t)__double2loint(v[i + n]));
			const auto hi = swap((uint32_t)__double2hiint(v[i]), (uint32_t)__double2hiint(v[i + n]));
			v[i] = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
		}
	};
	halves([](uint32_t a, uint32_t b) __attribute__((always_inline)) {
		return __builtin_amdgcn_permlane32_swap(a, b, false, false);
	}, K / 2);
	halves([](uint32_t a, uint32_t b) __attribute__((always_inline)) {
		return __builtin_amdgcn_permlane16_swap(a, b, false, false);
	}, K / 4);
#define TBTKX_ROTATE(N)                                                                           \
	_Pragma("unroll") for (int i = 0; i < K / 4; i++) v[i] += __hiloint2double(                \
	    __builtin_amdgcn_update_dpp(0, __double2hiint(v[i]), 0x120 + N, 0xf, 0xf, true),           \
	    __builtin_amdgcn_update_dpp(0, __double2loint(v[i]), 0x120 + N, 0xf, 0xf, true));
	TBTKX_ROTATE(8)
	TBTKX_ROTATE(4)
	TBTKX_ROTATE(2)
	TBTKX_ROTATE(1)
#undef TBTKX_ROTATE
}

struct RunArgs {
	const uint32_t *ecol;          // of the model
	const double *ev2;
	const uint64_t *pal;           // 256 values, kEmpty where unused
	int W, N, L, La, hq, ds, A, B, tb, Gt;
	int ncol, col0;                // the call's columns, the launch's first
	const int64_t *sites;          // per column, or null: random phases
	uint64_t seed;
	int S, M;                      // steps; moments (without dots)
	double2 *mu;                   // without dots: M per column
	double *part;                  // dots: [step][workgroup][kDots]
	void *xg;                      // 64 bytes each: [parity][team][N]
	uint32_t xg_bytes, epoch;
	uint32_t *err;
};

// NE entries beside the diagonal, R rows per thread. DOTS: 0 gathers moments, 1
// sums the doubling dots, 2 those of complex vectors (a column is a part).
template <int NE, int R, int DOTS>
__global__ __launch_bounds__(kT, 2) void block_resident(RunArgs a) {
	constexpr int AW = (NE + 1) / 2, CW = (NE + 3) / 4;
	__shared__ float4 x0[kWin], x1[kWin];   // columns 0-3 and 4-7
	__shared__ double pal[256];
	__shared__ double red[kT / 64][kDots];
	__shared__ int stop;
	const int t = threadIdx.x, N = a.N, L = a.L, hq = a.hq, ds = a.ds;
	const int team = (int)blockIdx.x / a.Gt;
	const Tile tile = tile_of(L, a.La, a.A, a.B, a.tb, (int)blockIdx.x - team * a.Gt);
	const Tile window = grown(tile, hq, ds), inside = grown(tile, -hq, -ds);
	const int win = area(window), own = area(tile), P = window.w;
	const int frame = a.Gt > 1 ? own - area(inside) : 0, ring = a.Gt > 1 ? win - own : 0;
	const int col0 = a.col0 + team * kCols;
	auto place = [&](Cell c) __attribute__((always_inline)) {
		return (c.a - window.a) * P + c.b - window.b;
	};
	auto row_in = [&](int p) __attribute__((always_inline)) -> int {
		const int q = p / P;
		const int64_t r = (int64_t)(window.a + q) * L + window.b + p - q * P;
		return r < 0 || r >= N ? -1 : (int)r;
	};
	// The palette first: the codes are looked up in it.
	for (int i = t; i < 256; i += kT) pal[i] = __longlong_as_double((long long)a.pal[i]);
	if (t == 0) stop = 0;
	__syncthreads();
	double diag[R];
	uint32_t adr[R][AW], code[R][CW];
	int pos[R];                    // window element, -1: no row
	float y[R][kCols];
#pragma unroll
	for (int j = 0; j < R; j++) {
		const int i = t + kT * j;
		pos[j] = -1;
		diag[j] = 0.0;
#pragma unroll
		for (int s = 0; s < AW; s++) adr[j][s] = 0;
#pragma unroll
		for (int s = 0; s < CW; s++) code[j][s] = 0;
#pragma unroll
		for (int c = 0; c < kCols; c++) y[j][c] = 0.0f;
		if (i >= own) continue;
		if (i < frame) {
			pos[j] = place(frame_cell(tile, i, hq, ds));
		} else {
			const Tile &in = a.Gt > 1 ? inside : tile;
			const int q = (i - frame) / in.w;
			pos[j] = place(Cell{in.a + q, in.b + (i - frame) - q * in.w});
		}
		const int r = row_in(pos[j]);
		const int64_t e = (int64_t)r * a.W;
		diag[j] = a.ev2[e];
#pragma unroll
		for (int u = 0; u < NE; u++) {
			uint32_t o = (uint32_t)pos[j];
			uint64_t k = 0;
			if (u + 1 < a.W) {
				const int off = (int)a.ecol[e + u + 1] - r;
				const int lay = !hq ? 0 : 2 * off > L ? 1 : 2 * off < -L ? -1 : 0;
				o = (uint32_t)(pos[j] + off - lay * (L - P));
				k = (uint64_t)__double_as_longlong(a.ev2[e + u + 1]);
			}
			uint32_t s = hash8(k);
			for (int i2 = 0; i2 < 256 && (uint64_t)__double_as_longlong(pal[s]) != k; i2++)
				s = (s + 1) & 255u;
			adr[j][u / 2] |= o << 16 * (u & 1);
			code[j][u / 4] |= s << 8 * (u & 3);
		}
	}
	// Start vectors.
	int site[kCols];
#pragma unroll
	for (int c = 0; c < kCols; c++)
		site[c] = DOTS != 2 && col0 + c < a.ncol ? (int)a.sites[col0 + c] : -1;
	for (int i = t; i < win; i += kT) {
		const int r = row_in(i);
		float v[kCols];
#pragma unroll
		for (int c = 0; c < kCols; c++) v[c] = r >= 0 && r == site[c] ? 1.0f : 0.0f;
		if (DOTS == 2 && r >= 0) {
#pragma unroll
			for (int c = 0; c < kCols; c += 2) {
				if (col0 + c >= a.ncol) break;
				const double2 z = random_phase(
				    a.seed, (uint64_t)((col0 + c) / 2) * (uint64_t)N + (uint64_t)r);
				v[c] = (float)z.x;
				v[c + 1] = (float)z.y;
			}
		}
		x0[i] = make_float4(v[0], v[1], v[2], v[3]);
		x1[i] = make_float4(v[4], v[5], v[6], v[7]);
	}
	// Without dots: this thread's column's start site, if it is in the tile.
	int mine = -1;
	if (!DOTS && t < kCols && col0 + t < a.ncol) {
		const int r = (int)a.sites[col0 + t], la = r / L, lb = r - la * L;
		if (la >= tile.a && la < tile.a + tile.h && lb >= tile.b && lb < tile.b + tile.w)
			mine = place(Cell{la, lb});
	}
	auto gather = [&](int n) __attribute__((always_inline)) {
		if (DOTS || mine < 0) return;
		const float *x = reinterpret_cast<const float *>(t < 4 ? x0 : x1);
		a.mu[(int64_t)(col0 + t) * a.M + n] = make_double2((double)x[4 * mine + (t & 3)], 0.0);
	};
	const __amdgpu_buffer_rsrc_t xg = __builtin_amdgcn_make_buffer_rsrc(a.xg, 0, a.xg_bytes, 0x00027000);
	const int teams = (int)gridDim.x / a.Gt;
	auto slot_of = [&](int n, int r) __attribute__((always_inline)) {
		return (uint32_t)((((n & 1) * teams + team) * (int64_t)N + r) * 4);
	};
	const int pf = t < frame ? row_in(pos[0]) : -1;
	// This thread's first two rows of the ring.
	int hp[2], hr[2];
#pragma unroll
	for (int i = 0; i < 2; i++) {
		hp[i] = t + kT * i < ring ? place(frame_cell(window, t + kT * i, hq, ds)) : -1;
		hr[i] = hp[i] < 0 ? -1 : row_in(hp[i]);
	}
	// Takes two rows of x_n into the window.
	auto take = [&](const int (&p)[2], const int (&r)[2], int n) __attribute__((always_inline)) {
		const uint32_t want = a.epoch + (uint32_t)n;
		const u32x4 none = {0, want, 0, want};
		u32x4 w[2][4];
		const long long begin = wall_clock64();
		int spins = 0;
		for (;;) {
			bool ok = true;
#pragma unroll
			for (int i = 0; i < 2; i++)
#pragma unroll
				for (int q = 0; q < 4; q++) {
					w[i][q] = none;
					if (r[i] >= 0) w[i][q] = get(xg, slot_of(n, r[i]) + q);
				}
#pragma unroll
			for (int i = 0; i < 2; i++)
#pragma unroll
				for (int q = 0; q < 4; q++) ok = ok && w[i][q].y == want && w[i][q].w == want;
			if (ok) break;
			if ((++spins & 63) == 0 &&
			    (wall_clock64() - begin > kWaitTicks ||
			     __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)) {
				__hip_atomic_store(a.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
				stop = 1;
				return;
			}
		}
#pragma unroll
		for (int i = 0; i < 2; i++) {
			if (r[i] < 0) continue;
			auto f = [](uint32_t v) __attribute__((always_inline)) { return __uint_as_float(v); };
			x0[p[i]] = make_float4(f(w[i][0].x), f(w[i][0].z), f(w[i][1].x), f(w[i][1].z));
			x1[p[i]] = make_float4(f(w[i][2].x), f(w[i][2].z), f(w[i][3].x), f(w[i][3].z));
		}
	};
	auto step = [&](auto first, int n) __attribute__((always_inline)) {
		constexpr bool FIRST = decltype(first)::value;
#pragma unroll
		for (int j = 0; j < R; j++) {
			// The packed words stay packed: unpacked once for all steps, they would
			// take more registers than there are.
#pragma unroll
			for (int s = 0; s < AW; s++) asm volatile("" : "+v"(adr[j][s]));
#pragma unroll
			for (int s = 0; s < CW; s++) asm volatile("" : "+v"(code[j][s]));
			asm volatile("" : "+v"(pos[j]));
			if (pos[j] < 0) continue;
			double acc[kCols], own8[kCols];
			auto read = [&](int p, double (&v)[kCols]) __attribute__((always_inline)) {
				const float4 lo = x0[p], hi = x1[p];
				v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w;
				v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
			};
			read(pos[j], own8);
#pragma unroll
			for (int c = 0; c < kCols; c++)
				acc[c] = fma(diag[j], own8[c], FIRST ? 0.0 : -(double)y[j][c]);
#pragma unroll
			for (int u = 0; u < NE; u++) {
				const double v = pal[code[j][u / 4] >> 8 * (u & 3) & 255u];
				double x[kCols];
				read((int)(adr[j][u / 2] >> 16 * (u & 1) & 0xffffu), x);
#pragma unroll
				for (int c = 0; c < kCols; c++) acc[c] = fma(v, x[c], acc[c]);
			}
#pragma unroll
			for (int c = 0; c < kCols; c++) {
				y[j][c] = (float)(FIRST ? 0.5 * acc[c] : acc[c]);
				asm volatile("" : "+v"(y[j][c]));   // kept as FP32, not also widened
			}
			if (kT * j < frame && t + kT * j < frame && n < a.S) {
				const uint32_t at = slot_of(n, j == 0 ? pf : row_in(pos[j])), tag = a.epoch + (uint32_t)n;
#pragma unroll
				for (int q = 0; q < 4; q++) {
					const u32x4 w = {__float_as_uint(y[j][2 * q]), tag, __float_as_uint(y[j][2 * q + 1]), tag};
					__builtin_amdgcn_raw_buffer_store_b128(w, xg, (at + q) * 16u, 0,
					                                       kCoherent | kVolatile);
				}
			}
		}
		__syncthreads();
		// x_n into the window, x_{n-1} into the registers, and their dots: here,
		// where no row's sums take registers.
		double d[2 * kCols], im[kCols / 2];
#pragma unroll
		for (int c = 0; c < 2 * kCols; c++) d[c] = 0.0;
#pragma unroll
		for (int c = 0; c < kCols / 2; c++) im[c] = 0.0;
#pragma unroll
		for (int j = 0; j < R; j++) {
			asm volatile("" : "+v"(pos[j]));
			if (pos[j] < 0) continue;
			const float4 lo = x0[pos[j]], hi = x1[pos[j]];
			x0[pos[j]] = make_float4(y[j][0], y[j][1], y[j][2], y[j][3]);
			x1[pos[j]] = make_float4(y[j][4], y[j][5], y[j][6], y[j][7]);
			const float old[kCols] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
			for (int c = 0; c < kCols && DOTS; c++) {
				d[c] = fma((double)old[c], (double)old[c], d[c]);
				d[kCols + c] = fma((double)y[j][c], (double)old[c], d[kCols + c]);
			}
#pragma unroll
			for (int c = 0; c < kCols && DOTS == 2; c += 2) {
				im[c / 2] = fma((double)y[j][c], (double)old[c + 1], im[c / 2]);
				im[c / 2] = fma(-(double)y[j][c + 1], (double)old[c], im[c / 2]);
			}
			// A row's dots end with it: put off, they would keep all rows' values.
#pragma unroll
			for (int c = 0; c < 2 * kCols && DOTS; c++) asm volatile("" : "+v"(d[c]));
#pragma unroll
			for (int c = 0; c < kCols; c++) {
				y[j][c] = old[c];
				asm volatile("" : "+v"(y[j][c]));
			}
		}
		if (DOTS) {
			const int row = (t & 63) >> 4;
			wave_sums<2 * kCols>(d);
			if ((t & 15) == 0)
#pragma unroll
				for (int i = 0; i < kCols / 2; i++)
					red[t >> 6][i + kCols * (row >> 1) + kCols / 2 * (row & 1)] = d[i];
			if (DOTS == 2) {
				wave_sums<kCols / 2>(im);
				if ((t & 15) == 0) red[t >> 6][2 * kCols + row] = im[0];
			}
		}
		if (n < a.S && ring > 0) {
			take(hp, hr, n);
			for (int i = t + 2 * kT; i < ring; i += 2 * kT) {
				int p[2], r[2];
#pragma unroll
				for (int q = 0; q < 2; q++) {
					p[q] = i + kT * q < ring ? place(frame_cell(window, i + kT * q, hq, ds)) : -1;
					r[q] = p[q] < 0 ? -1 : row_in(p[q]);
				}
				take(p, r, n);
			}
		}
		__syncthreads();
		if (DOTS && t < kDots && (t < 2 * kCols || DOTS == 2)) {
			double s = 0.0;
#pragma unroll
			for (int w = 0; w < kT / 64; w++) s += red[w][t];
			a.part[((int64_t)(n - 1) * gridDim.x + blockIdx.x) * kDots + t] = s;
		}
	};
	__syncthreads();
	gather(0);
	if (a.S < 1) return;
	step(std::true_type{}, 1);
	if (stop) return;
	gather(1);
	for (int n = 2; n <= a.S; n++) {
		step(std::false_type{}, n);
		if (stop) return;
		gather(n);
	}
}

// D[team][step][k] = sum over the team's workgroups, in their order.
__global__ __launch_bounds__(kThreads) void block_dots(const double *__restrict__ part,
                                                       double *__restrict__ D, int S, int teams,
                                                       int Gt, int nk) {
	const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
	if (i >= (int64_t)S * teams * kDots) return;
	const int k = (int)(i % kDots), n = (int)(i / kDots % S), team = (int)(i / kDots / S);
	double s = 0.0;
	if (k < nk) {
		const double *p = part + ((int64_t)n * teams * Gt + (int64_t)team * Gt) * kDots + k;
		for (int g = 0; g < Gt; g++) s += p[(int64_t)g * kDots];
	}
	D[i] = s;
}

// Times in us of the rule in resident_block: a step of one round of 512 rows with
// one entry beside the diagonal; a call, a cooperative launch, a launch's setup per
// round (entries and codes), the sum of its dots per workgroup of a team; and
// the share of the step kernels' time to beat. Model and measured, whole calls: 1,024,000
// states, 64 columns in 8 passes, 2 steps gathered 520 509, 4 with dots 1270 1290; 159,520
// states, 37 columns, 30 steps with dots 350 343; 1800 states, 64 columns, 20 steps
// with dots 137 116.
constexpr double kRound = 0.11, kStep = 0.6;
constexpr double kLeastStep = kStep + kRound * (1 + 2);
constexpr double kCall = 50, kLaunch = 17, kSetup = 3, kSumDots = 0.3, kWorth = 0.9;

typedef BlockShape Shape;

// The tiles and teams of the least time for V columns of a model; us = 0: none.
// Time of a step in us: rounds of 512 rows, the ring's bytes and its passes; model
// and measured per pass: 2.0 2.1 (900 rows in one workgroup), 3.4 2.5 (1600), 7.3 6.6
// (250,000 rows in tiles), 8.2 8.6 (159,520), 10.7 11.9 (1,048,576).
Shape shape_of(int64_t N, int ne, int layer, int reach, int64_t band, int V, int cus) {
	Shape best;
	const int groups = (V + kCols - 1) / kCols;
	auto consider = [&](int64_t L, int64_t hq, int64_t ds, int64_t ta, int64_t tb) {
		const int64_t La = N / L, A = (La + ta - 1) / ta, B = (L + tb - 1) / tb, Gt = ta * tb;
		if ((La + A - 1) / A != ta || (L + B - 1) / B != tb) return;
		const int64_t low = La - (ta - 1) * A, narrow = L - (tb - 1) * B;
		if (Gt > 1 && (low < 2 * hq || narrow < 2 * ds || A < 2 * hq || B < 2 * ds)) return;
		const int64_t own = A * B, win = (A + 2 * hq) * (B + 2 * ds);
		if (win > kWin || own > kMaxRows * kT) return;
		const int64_t fit = std::min<int64_t>(cus / Gt, groups);
		if (fit < 1) return;
		const int64_t passes = (groups + fit - 1) / fit, teams = (groups + passes - 1) / passes;
		const double rounds = (double)((own + kT - 1) / kT);
		double us = kStep + rounds * kRound * (ne + 2);
		if (Gt > 1)
			us += 1.6 + (double)(teams * Gt * (win - own)) * 128 / 8e6 +
			      0.7 * (double)((win - own - 1) / (2 * kT));
		us *= (double)passes;
		if (best.us == 0 || us < best.us) {
			best.L = (int)L, best.hq = (int)hq, best.ds = (int)ds;
			best.A = (int)A, best.B = (int)B, best.Gt = (int)Gt;
			best.teams = (int)teams, best.passes = (int)passes;
			best.rounds = (int)((own + kT - 1) / kT);
			best.us = us;
		}
	};
	if (N <= kMaxRows * kT) consider(N, 0, 0, 1, 1);
	if (N > (int64_t)cus * kMaxRows * kT) return best;
	if (layer)
		for (int64_t ta = 1; ta <= std::min<int64_t>(cus, N / layer); ta++)
			for (int64_t tb = 1; tb * ta <= cus; tb++)
				if (ta * tb > 1) consider(layer, 1, reach, ta, tb);
	if (band < N)
		for (int64_t tb = 2; tb <= cus; tb++) consider(N, 0, band, 1, tb);
	return best;
}

template <int NE, int DOTS>
const void *kernel_rows(int rows) {
	return rows <= 1   ? (const void *)block_resident<NE, 1, DOTS>
	       : rows <= 2 ? (const void *)block_resident<NE, 2, DOTS>
	       : rows <= 4 ? (const void *)block_resident<NE, 4, DOTS>
	       : rows <= 6 ? (const void *)block_resident<NE, 6, DOTS>
	                   : (const void *)block_resident<NE, 8, DOTS>;
}
template <int DOTS>
const void *kernel_of(int ne, int rows) {
	switch (ne) {
	case 1:
	case 2:
	case 3: return kernel_rows<3, DOTS>(rows);
	case 4: return kernel_rows<4, DOTS>(rows);
	case 5: return kernel_rows<5, DOTS>(rows);
	case 6: return kernel_rows<6, DOTS>(rows);
	default: return kernel_rows<7, DOTS>(rows);
	}
}

// Palettes, entries per row and lattice views of the call's models, once per
// generation.
int scan_models(tbtkx_context *h, const BlockCall &c, tbtkx_context::BlockForms &f) {
	if (f.gen == c.gen && (int)f.ne.size() == c.K) return TBTKX_OK;
	int rc;
	f.gen = -1;
	f.shapes.clear();
	const size_t at = (size_t)c.K * sizeof(Scan);
	if ((rc = f.scan.reserve(at + (size_t)c.K * sizeof(ScanModel)))) return rc;
	std::vector<ScanModel> sm(c.K);
	int64_t most = 1;
	for (int m = 0; m < c.K; m++) {
		sm[m] = ScanModel{c.N[m], c.e0[m], c.W[m], 0};
		most = std::max(most, c.N[m]);
	}
	Scan *dev = f.scan.as<Scan>();
	ScanModel *dm = reinterpret_cast<ScanModel *>(f.scan.as<char>() + at);
	TBTKX_CHECK_HIP(hipMemcpyAsync(dm, sm.data(), sm.size() * sizeof(ScanModel),
	                               hipMemcpyHostToDevice, h->stream));
	scan_init<<<c.K, kThreads, 0, h->stream>>>(dev);
	const unsigned gx = (unsigned)std::min<int64_t>(512, (most + 4 * kThreads - 1) / (4 * kThreads));
	scan_model<<<dim3(gx, c.K), kThreads, 0, h->stream>>>(dm, c.ecol, c.ev2, dev);
	TBTKX_CHECK_HIP(hipGetLastError());
	std::vector<Scan> host(c.K);
	TBTKX_CHECK_HIP(hipMemcpyAsync(host.data(), dev, at, hipMemcpyDeviceToHost, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	f.ne.assign(c.K, 0);
	f.layer.assign(c.K, 0);
	f.reach.assign(c.K, 0);
	std::vector<uint8_t> seen(65536);
	for (int m = 0; m < c.K; m++) {
		if (host[m].bad) continue;
		f.ne[m] = std::max<int>(1, (int)host[m].ne);
		for (int o = 0; o < 65536; o++) seen[o] = host[m].seen[o >> 5] >> (o & 31) & 1;
		layer_stride(c.N[m], seen, &f.layer[m], &f.reach[m]);
	}
	f.gen = c.gen;
	return TBTKX_OK;
}

}  // namespace

int resident_block(tbtkx_context *h, const BlockCall &c, double *out, bool *done) {
	*done = false;
	// Against the step kernels. Wide rings lose: 864,000 states (96 x 100 x 90), 64
	// columns, a ring of 4000 of 3800 rows, 270 us a step against 173; and so do many passes
	// of few steps: 1,024,000 states, 64 columns in 8 passes, 4 steps with dots 1287 us
	// against 833, 10 steps 1668 against 1920.
	int64_t vectors = 0;
	std::vector<int> S(c.K);
	double least = kCall;
	for (int m = 0; m < c.K; m++) {
		S[m] = c.doubling ? (c.M[m] + 1) / 2 : c.M[m] - 1;
		if (S[m] < 1) return TBTKX_OK;
		vectors += c.cols[m];
		least += kLeastStep * S[m] + kLaunch + kSetup;
	}
	// A launch per model and its shortest steps cost more already: no scan, which
	// takes 10 KB and some 50 us of the host per model (a batch of 1000 small models).
	if (least > kWorth * c.theirs) return TBTKX_OK;
	int rc;
	if (!cooperative_now(h)) return TBTKX_OK;
	// No memory for this path's own scratch: the step kernels need what it holds.
	auto no_memory = [&]() {
		(void)hipGetLastError();
		for (tbtkx::DevBuf *b : {&h->res_xg, &h->rb_part, &h->rb_D}) b->release();
		return TBTKX_OK;
	};
	tbtkx_context::BlockForms &f = c.single ? h->rb_single : h->rb_multi;
	if ((rc = scan_models(h, c, f))) return rc == TBTKX_ERR_OOM ? no_memory() : rc;
	std::vector<Shape> sh(c.K);
	double mine = kCall;
	int64_t steps = 0;
	for (int m = 0; m < c.K; m++) {
		if (!f.ne[m]) return TBTKX_OK;
		const auto key = std::make_pair(m, c.cols[m]);
		auto known = f.shapes.find(key);
		if (known == f.shapes.end()) {
			if (f.shapes.size() >= 4096) f.shapes.clear();
			known = f.shapes.emplace(key, shape_of(c.N[m], f.ne[m], f.layer[m], f.reach[m], c.band[m],
			                                       c.cols[m], h->num_cus)).first;
		}
		sh[m] = known->second;
		if (sh[m].us == 0) return TBTKX_OK;
		// Dots of complex vectors: 12.8 us where the model gives 9.4.
		steps += (int64_t)S[m] * sh[m].passes;
		mine += sh[m].us * (c.phases ? 1.35 : 1.0) * S[m] +
		        sh[m].passes * (kLaunch + kSetup * sh[m].rounds + (c.doubling ? kSumDots * sh[m].Gt : 0.0));
	}
	if (mine > kWorth * c.theirs) return TBTKX_OK;

	size_t part = 0, D = 0, xg = 0, mu = 0;
	uint32_t phases = 0;
	std::vector<size_t> off(c.K), out_off(c.K);
	size_t o = 0;
	for (int m = 0; m < c.K; m++) {
		const Shape &s = sh[m];
		const size_t groups = (size_t)s.passes * s.teams;
		off[m] = c.doubling ? D : mu;
		D += groups * S[m] * kDots;
		mu += (size_t)c.cols[m] * c.M[m];
		out_off[m] = o;
		o += (size_t)(c.phases ? c.cols[m] / 2 : c.cols[m]) * c.M[m];
		part = std::max(part, (size_t)S[m] * s.teams * s.Gt * kDots * 8);
		if (s.Gt > 1) xg = std::max(xg, (size_t)2 * s.teams * c.N[m] * 64);
		phases += (uint32_t)s.passes * (uint32_t)(S[m] + 2);
	}
	// Long calls keep to the step kernels rather than to gigabytes of scratch.
	if (part > ((size_t)1 << 30) || xg >= ((size_t)1 << 32) - 64 || phases > (1u << 30))
		return TBTKX_OK;
	if ((rc = exchange_buffer(h, xg, phases))) return rc == kDeclined ? no_memory() : rc;
	const size_t res_bytes = c.doubling ? D * 8 : mu * 16;
	if ((c.doubling && (rc = h->rb_part.reserve(part))) || (rc = h->rb_D.reserve(res_bytes)))
		return rc == TBTKX_ERR_OOM ? no_memory() : rc;
	if (c.sites) {
		if ((rc = h->rb_sites.reserve((size_t)vectors * 8)))
			return rc == TBTKX_ERR_OOM ? no_memory() : rc;
		TBTKX_CHECK_HIP(hipMemcpyAsync(h->rb_sites.ptr, c.sites, (size_t)vectors * 8,
		                               hipMemcpyHostToDevice, h->stream));
	}
	TBTKX_CHECK_HIP(hipEventRecord(h->ev_start, h->stream));
	int64_t site0 = 0;
	for (int m = 0; m < c.K; m++) {
		const Shape &s = sh[m];
		RunArgs a{};
		a.ecol = c.ecol + c.e0[m];
		a.ev2 = c.ev2 + c.e0[m];
		a.pal = f.scan.as<Scan>()[m].key;
		a.W = c.W[m];
		a.N = (int)c.N[m];
		a.L = s.L;
		a.La = (int)(c.N[m] / s.L);
		a.hq = s.hq;
		a.ds = s.ds;
		a.A = s.A;
		a.B = s.B;
		a.tb = (s.L + s.B - 1) / s.B;
		a.Gt = s.Gt;
		a.ncol = c.cols[m];
		a.sites = c.sites ? h->rb_sites.as<int64_t>() + site0 : nullptr;
		a.seed = c.seed;
		a.S = S[m];
		a.M = c.M[m];
		a.mu = c.doubling ? nullptr : h->rb_D.as<double2>() + off[m];
		a.part = h->rb_part.as<double>();
		a.xg = h->res_xg.ptr;
		a.xg_bytes = (uint32_t)xg;
		a.err = h->res_err.as<uint32_t>();
		const void *k = c.phases      ? kernel_of<2>(f.ne[m], s.rounds)
		                : c.doubling ? kernel_of<1>(f.ne[m], s.rounds)
		                             : kernel_of<0>(f.ne[m], s.rounds);
		for (int p = 0; p < s.passes; p++) {
			a.col0 = p * s.teams * kCols;
			const int left = (c.cols[m] - a.col0 + kCols - 1) / kCols, teams = std::min(s.teams, left);
			a.epoch = h->res_epoch;
			h->res_epoch += (uint32_t)(S[m] + 2);
			void *args[] = {&a};
			if (launch_cooperative(h, k, (unsigned)(teams * s.Gt), kT, args)) return TBTKX_OK;
			if (!c.doubling) continue;
			const int64_t n = (int64_t)S[m] * teams * kDots;
			block_dots<<<(unsigned)((n + kThreads - 1) / kThreads), kThreads, 0, h->stream>>>(
			    a.part, h->rb_D.as<double>() + off[m] + (size_t)p * s.teams * S[m] * kDots, S[m], teams,
			    s.Gt, c.phases ? kDots : 2 * kCols);
			TBTKX_CHECK_HIP(hipGetLastError());
		}
		site0 += c.cols[m];
	}
	TBTKX_CHECK_HIP(hipEventRecord(h->ev_stop, h->stream));
	std::vector<double> res(res_bytes / 8);
	TBTKX_CHECK_HIP(hipMemcpyAsync(res.data(), h->rb_D.ptr, res_bytes, hipMemcpyDeviceToHost, h->stream));
	bool given_up = false;
	if ((rc = exchange_given_up(h, &given_up))) return rc;
	if (given_up) return TBTKX_OK;
	float ms = 0;
	TBTKX_CHECK_HIP(hipEventElapsedTime(&ms, h->ev_start, h->ev_stop));
	h->last_ms = ms;
	h->last_launches = steps;
	h->last_resident = 1;
	*done = true;
	if (!c.doubling) {
		memcpy(out, res.data(), res_bytes);
		return TBTKX_OK;
	}
	for (int m = 0; m < c.K; m++) {
		const int per = c.phases ? 2 : 1, M = c.M[m];
		for (int v = 0; v * per < c.cols[m]; v++) {
			const int col = v * per, k = col % kCols;
			const double *d = res.data() + off[m] + (size_t)(col / kCols) * S[m] * kDots;
			double *o2 = out + 2 * (out_off[m] + (size_t)v * M);
			double mu0 = 0, mu1 = 0, im1 = 0;
			for (int n = 0; n < S[m]; n++, d += kDots) {
				const double d0 = c.phases ? d[k] + d[k + 1] : d[k];
				const double d1 = c.phases ? d[kCols + k] + d[kCols + k + 1] : d[kCols + k];
				const double im = c.phases ? d[2 * kCols + k / 2] : 0.0;
				if (n == 0) mu0 = d0, mu1 = d1, im1 = im;
				o2[4 * n] = n ? 2 * d0 - mu0 : mu0;
				o2[4 * n + 1] = 0.0;
				if (2 * n + 1 < M) {
					o2[4 * n + 2] = n ? 2 * d1 - mu1 : mu1;
					o2[4 * n + 3] = n ? 2 * im - im1 : im1;
				}
			}
		}
	}
	return TBTKX_OK;
}

}  // namespace tbtkx
