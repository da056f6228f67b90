// Lookup table and FP64 Green's-function contraction.
//
// Table (Lib/src/Solver/ChebyshevExpander.cpp:256-268), E~ = E_e/s:
//   L[n][e] = (1/s) * (-2i/sqrt(1 - E~^2)) * exp(-i n acos E~) / (n == 0 ? 2 : 1)
// Contraction (Lib/src/Solver/ChebyshevExpander.cpp:324-370), n ascending:
//   Retarded      G += L*c            Advanced     G += c*conj(L)
//   Principal     G += -c*Re(L)       NonPrincipal G -= (c*i)*Im(L)
// The FP64 kernels keep that order and operation sequence (no fused
// multiply-add), so with an uploaded host table they reproduce the reference
// bit for bit; with the device-generated table the difference is that of
// the device acos/sqrt/sincos against the host libm (a few ulp).
//
// It is an FP64 GEMV/GEMM of 8 K M E flops whose sums run serially over n.
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "host_math.hpp"

namespace tbtkx {
namespace {

__global__ __launch_bounds__(kThreads) void lut_generate(
    double2 *__restrict__ L, int M, int E, double lo, double dx, double s) {
#pragma clang fp contract(off)
	const int e = blockIdx.x * kThreads + threadIdx.x;
	const int n = blockIdx.y;
	if (e >= E) return;
	const double En = (lo + e * dx) / s;
	const double r = sqrt(1 - En * En);
	// (1/s) * ((-0, -2) / r)
	const double ar = (-2.0 * 0.0 / r) * (1 / s);
	const double ai = (-2.0 / r) * (1 / s);
	double sn, cs;
	sincos((-1.0 * (double)n) * acos(En), &sn, &cs);
	const double denom = n == 0 ? 2.0 : 1.0;
	L[(int64_t)n * E + e] = make_double2((ar * cs - ai * sn) / denom,
	                                     (ar * sn + ai * cs) / denom);
}

// Damping of K coefficient vectors C[k*M + n] in FP64, in place; one thread
// per moment n computes its factor once and walks the vectors.
//   Lorentz (Lib/src/Solver/ChebyshevExpander.cpp:190-196; the reference's
//   GPU path damps on the device too, Lib/src/cuda/ChebyshevSolver.cu:632-645):
//     c *= sinh(lambda (1 - n/M)); c /= sinh(lambda), lambda = broadening*M,
//     real and imaginary part each, as std::complex<double> * and / double do.
//   Jackson (Weisse et al., Rev. Mod. Phys. 78, 275 (2006), eq. 71):
//     g_n = ((M - n + 1) cos(q n) + sin(q n) cos(q) / sin(q)) / (M + 1),
//     q = pi/(M + 1); c *= g_n.
__global__ __launch_bounds__(kThreads) void damp_coeffs(double2 *__restrict__ C, int K, int M,
                                                        int kind, double broadening) {
#pragma clang fp contract(off)
	const int n = blockIdx.x * kThreads + threadIdx.x;
	if (n >= M) return;
	double num, den;
	if (kind == TBTKX_DAMP_LORENTZ) {
		const double lambda = broadening * M;
		num = sinh(lambda * (1 - n / (double)M));
		den = sinh(lambda);
	} else {
		const double q = M_PI / (M + 1);
		num = (double)(M - n + 1) * cos(q * n) + sin(q * n) * cos(q) / sin(q);
		den = (double)(M + 1);
	}
	const double g = num / den;
	for (int k = blockIdx.y; k < K; k += gridDim.y) {
		double2 c = C[(int64_t)k * M + n];
		if (kind == TBTKX_DAMP_LORENTZ) {
			c.x = (c.x * num) / den;
			c.y = (c.y * num) / den;
		} else {
			c.x = c.x * g;
			c.y = c.y * g;
		}
		C[(int64_t)k * M + n] = c;
	}
}

// Direct evaluation without a table, Lib/src/Solver/ChebyshevExpander.cpp:
// 371-432: per energy E~ = E/s, theta = acos(E~),
//   Retarded     (c0/2 + sum_n c_n e^{-in theta}) * (-2i/s)
//   Advanced     (c0/2 + sum_n conj(c_n e^{-in theta})) * (2i/s)
//   Principal    (sum_n c_n sin(n theta)) * (2/s)
//   NonPrincipal (c0/2 + sum_n c_n cos(n theta)) * (2i/s)
// all divided by sqrt(1 - E~^2); energies e0 + e*de as Range::operator[].
// The trigonometric factors come from the host's libm (direct_factors), the
// functions the reference calls, so the sums below reproduce its results bit
// for bit: the factor array holds e^{-in theta} as (re, im) pairs (Retarded,
// Advanced), sin(n theta) (Principal) or cos(n theta) (NonPrincipal) at
// [(n-1)*E + e], and den[e] = sqrt(1 - E~^2).

// One term of either contraction, with the values of the reference's operation
// order. Real and imaginary part never mix, and each is a sum of
//   g + (l.x p - l.y q)   (Retarded, Advanced)   or   g + l p
// with (p, q) made of the coefficient and the type by exact operations:
//   Retarded  re (c.x, c.y)    im (c.y, -c.x)
//   Advanced  re (c.x, -c.y)   im (c.y, c.x), direct: re (c.x, c.y), im (-c.y, c.x)
//   Principal re -c.x, im -c.y, direct: c.x, c.y
//   NonPrincipal  -(c * i), (c * i) = (cr*0 - ci*1, cr*1 + ci*0); direct: c.x, c.y
// F: the part of the table or factor array that the type reads.
template <int TYPE, bool DIRECT>
struct Term {
	static constexpr bool kPair = TYPE == TBTKX_RETARDED || TYPE == TBTKX_ADVANCED;
	typedef typename std::conditional<kPair, double2, double>::type F;
	static constexpr int kFirst = DIRECT ? 1 : 0;   // first n of the sum

	__device__ __forceinline__ static F load(const double *t, int64_t at) {
		if constexpr (kPair) return reinterpret_cast<const double2 *>(t)[at];
		else if constexpr (DIRECT) return t[at];
		else return t[2 * at + (TYPE == TBTKX_PRINCIPAL ? 0 : 1)];
	}
	// The same through a buffer resource. `row` is a scalar offset, which the
	// resource's bounds check leaves out: it must lie inside the array.
	static constexpr int kBytes = DIRECT && !kPair ? 8 : 16;   // of an array element
	static constexpr int kPart = !DIRECT && TYPE == TBTKX_NONPRINCIPAL ? 8 : 0;
	__device__ __forceinline__ static F load(__amdgpu_buffer_rsrc_t t, uint32_t lane, uint32_t row) {
		if constexpr (kPair)
			return __builtin_bit_cast(double2, __builtin_amdgcn_raw_buffer_load_b128(t, lane, row, 0));
		else
			return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(t, lane + kPart, row, 0));
	}
	__device__ __forceinline__ static double start(double c0) {
		return DIRECT && TYPE != TBTKX_PRINCIPAL ? c0 / 2. : 0.0;
	}
	// The real part's (p, q); without kPair the real and imaginary part's p.
	__device__ __forceinline__ static double2 prepare(double2 c) {
#pragma clang fp contract(off)
		if constexpr (kPair) return TYPE == TBTKX_ADVANCED && !DIRECT ? make_double2(c.x, -c.y) : c;
		else if constexpr (DIRECT) return c;
		else if constexpr (TYPE == TBTKX_PRINCIPAL) return make_double2(-c.x, -c.y);
		else return make_double2(-(c.x * 0.0 - c.y * 1.0), -(c.x * 1.0 + c.y * 0.0));
	}
	// The imaginary part's (p, q) from the prepared coefficient.
	__device__ __forceinline__ static double2 imag(double2 c) {
		if constexpr (!kPair) return make_double2(c.y, 0.0);
		else if constexpr (TYPE == TBTKX_RETARDED) return make_double2(c.y, -c.x);
		else return make_double2(-c.y, c.x);
	}
	__device__ __forceinline__ static double add(F l, double2 c, double g) {
#pragma clang fp contract(off)
		if constexpr (kPair) return g + (l.x * c.x - l.y * c.y);
		else return g + l * c.x;
	}
	// The finished value: the direct form's prefactor and denominator.
	__device__ __forceinline__ static double2 finish(double gr, double gi, double den, double s) {
#pragma clang fp contract(off)
		if constexpr (!DIRECT) return make_double2(gr, gi);
		double hr, hi;
		if constexpr (TYPE == TBTKX_PRINCIPAL) {
			const double fr = 2. / s;
			hr = gr * fr;
			hi = gi * fr;
		} else {
			const double fr = TYPE == TBTKX_RETARDED ? -2. * 0.0 / s : 2. * 0.0 / s;
			const double fi = TYPE == TBTKX_RETARDED ? -2. / s : 2. / s;
			hr = gr * fr - gi * fi;
			hi = gr * fi + gi * fr;
		}
		return make_double2(hr / den, hi / den);
	}
};

// Few vectors: every sum is a serial chain over n, and there are only K E of
// them, so the time is the chain, and the latency and per-CU rate of the
// table's rows. A wavefront takes 16 energies, both parts and two vectors (a lane
// each), which spreads the rows over four times the CUs that 64 energies a
// wavefront would use, with kAhead rows loaded while the kAhead before them are
// added; the lanes' (p, q) come from LDS, kFewChunk terms at a time.
// 1000 energies, 1000 moments, 4 vectors (direct): a thread per energy with 16
// rows ahead took 52 us.
constexpr int kFewChunk = 512;

template <int TYPE, bool DIRECT>
__global__ __launch_bounds__(64) void contract_few(
    const double *__restrict__ L, const double2 *__restrict__ C, const double *__restrict__ den,
    double2 *__restrict__ G, int K, int M, int E, double s) {
	typedef Term<TYPE, DIRECT> O;
	typedef typename O::F F;
	constexpr int kAhead = O::kPair ? 16 : 32;
	__shared__ double2 sc[kFewChunk][4];   // vector, then real and imaginary part
	const int lane = threadIdx.x;
	const int e = blockIdx.x * 16 + (lane & 15);
	const int ec = e < E ? e : E - 1;
	const int im = (lane >> 4) & 1, v = lane >> 5;
	const int k0 = 2 * blockIdx.y, kv = k0 + v < K ? k0 + v : K - 1;
	// Row r of the array is term n = r + kFirst.
	const int rows = M - O::kFirst;
	const double2 c0 = C[(int64_t)kv * M];
	double g = O::start(im ? c0.y : c0.x);
	const double *const mine = reinterpret_cast<const double *>(&sc[0][lane >> 4]);
	const uint32_t rowb = (uint32_t)E * O::kBytes, off = (uint32_t)ec * O::kBytes;
	for (int r0 = 0; r0 < rows; r0 += kFewChunk) {
		const int n = rows - r0 < kFewChunk ? rows - r0 : kFewChunk;
		// The chunk's rows. A row takes a scalar add, a scalar minimum and one load,
		// where a lone wavefront pays every instruction in full. Rows read ahead of
		// the chunk's end repeat its last. Offsets stay in 32 bits: contract_launch
		// comes here with at most 16 x 4 energies per CU (16,384), 16 B each, and r
		// runs to 512 + 3 kAhead rows.
		const __amdgpu_buffer_rsrc_t tab = __builtin_amdgcn_make_buffer_rsrc(
		    const_cast<char *>(reinterpret_cast<const char *>(L)) + (int64_t)r0 * rowb, 0,
		    (uint32_t)n * rowb, 0x00027000);
		const uint32_t last = (uint32_t)(n - 1) * rowb;
		auto load = [&](F (&f)[kAhead], int r) __attribute__((always_inline)) {
#pragma unroll
			for (int i = 0; i < kAhead; i++) {
				const uint32_t row = (uint32_t)(r + i) * rowb;
				f[i] = O::load(tab, off, row < last ? row : last);
			}
		};
		F a[kAhead], b[kAhead];
		load(a, 0);
		__syncthreads();
		for (int i = lane; i < 2 * n; i += 64) {
			const int w = i >= n, q = w ? i - n : i;
			const double2 p =
			    O::prepare(C[(int64_t)(k0 + w < K ? k0 + w : K - 1) * M + r0 + q + O::kFirst]);
			sc[q][2 * w] = p;
			sc[q][2 * w + 1] = O::imag(p);
		}
		__syncthreads();
		auto add = [&](F (&f)[kAhead], int r) __attribute__((always_inline)) {
			// All of the batch's (p, q) first, or every pair of terms would wait
			// for its own LDS round trip.
			double p[kAhead], q[O::kPair ? kAhead : 1];
#pragma unroll
			for (int i = 0; i < kAhead; i++) {
				p[i] = mine[(r + i) * 8];
				if (O::kPair) q[i] = mine[(r + i) * 8 + 1];
			}
			__builtin_amdgcn_sched_barrier(0);
			if (r + kAhead <= n) {
#pragma unroll
				for (int i = 0; i < kAhead; i++)
					g = O::add(f[i], make_double2(p[i], O::kPair ? q[i] : 0.0), g);
			} else {
#pragma unroll
				for (int i = 0; i < kAhead; i++)
					if (r + i < n) g = O::add(f[i], make_double2(p[i], O::kPair ? q[i] : 0.0), g);
			}
		};
		for (int r = 0; r < n; r += 2 * kAhead) {
			load(b, r + kAhead);
			add(a, r);
			load(a, r + 2 * kAhead);
			if (r + kAhead < n) add(b, r + kAhead);
		}
	}
	// The lane of the real part takes the imaginary part from its neighbour.
	const double gi = __shfl(g, lane + 16);
	if (!im && e < E && k0 + v < K)
		G[(int64_t)(k0 + v) * E + e] = O::finish(g, gi, DIRECT ? den[e] : 0.0, s);
}

// Many vectors: a wavefront takes KT of them at 64 energies, so a table row
// is loaded once for KT vectors, and the four wavefronts of a workgroup share the
// row through L1. The coefficients of the workgroup's 4 KT vectors come
// prepared from LDS, kManyChunk terms at a time in two stages (one broadcast read
// per term and vector; as scalar loads, 16 B per term, they left the FP64 units
// idle two thirds of the time). Bound by FP64 issue: 8 operations per complex term
// (4 for the half-complex types).
template <int TYPE, bool DIRECT, int KT>
__global__ __launch_bounds__(kThreads) void contract_many(
    const double *__restrict__ L, const double2 *__restrict__ C, const double *__restrict__ den,
    double2 *__restrict__ G, int K, int M, int E, double s) {
	typedef Term<TYPE, DIRECT> O;
	typedef typename O::F F;
	constexpr int kAhead = 8, KW = 4 * KT, kManyChunk = 16;
	constexpr int kPer = KW * kManyChunk / kThreads;   // coefficients a thread stages
	static_assert(kPer >= 1 && kManyChunk % kAhead == 0, "staging split");
	__shared__ double2 sc[2][kManyChunk][KW];
	const int lane = threadIdx.x & 63;
	const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const int kb = blockIdx.y * KW, k0 = kb + wave * KT;
	const int e = blockIdx.x * 64 + lane;
	const int ec = e < E ? e : E - 1;
	const int rows = M - O::kFirst;
	// This thread stages terms n0 .. n0 + kPer - 1 of vector kb + ks; vectors and
	// terms past the end repeat the last.
	const int ks = threadIdx.x * kPer / kManyChunk, n0 = threadIdx.x * kPer % kManyChunk;
	const double2 *cs = C + (int64_t)(kb + ks < K ? kb + ks : K - 1) * M + O::kFirst;
	double2 st[kPer];
	auto fetch = [&](int r) __attribute__((always_inline)) {
#pragma unroll
		for (int i = 0; i < kPer; i++) {
			const int q = r + n0 + i;
			st[i] = cs[q < rows ? q : rows - 1];
		}
	};
	auto stage = [&](int b) __attribute__((always_inline)) {
#pragma unroll
		for (int i = 0; i < kPer; i++) sc[b][n0 + i][ks] = O::prepare(st[i]);
	};
	double gr[KT], gi[KT];
#pragma unroll
	for (int k = 0; k < KT; k++) {
		const double2 c0 = C[(int64_t)(k0 + k < K ? k0 + k : K - 1) * M];
		gr[k] = O::start(c0.x);
		gi[k] = O::start(c0.y);
	}
	auto load = [&](F (&v)[kAhead], int r) __attribute__((always_inline)) {
#pragma unroll
		for (int i = 0; i < kAhead; i++) {
			const int q = r + i < rows ? r + i : rows - 1;
			v[i] = O::load(L, (int64_t)q * E + ec);
		}
	};
	if (rows > 0) {
		F a[kAhead], b[kAhead];
		fetch(0);
		load(a, 0);
		stage(0);
		__syncthreads();
		int buf = 0;
		for (int r0 = 0; r0 < rows; r0 += kManyChunk, buf ^= 1) {
			if (r0 + kManyChunk < rows) fetch(r0 + kManyChunk);
#pragma unroll
			for (int h = 0; h < kManyChunk; h += kAhead) {
				load(b, r0 + h + kAhead);
#pragma unroll
				for (int i = 0; i < kAhead; i++) {
					if (r0 + h + i >= rows) break;
#pragma unroll
					for (int k = 0; k < KT; k++) {
						const double2 cn = sc[buf][h + i][wave * KT + k];
						gr[k] = O::add(a[i], cn, gr[k]);
						gi[k] = O::add(a[i], O::imag(cn), gi[k]);
					}
				}
#pragma unroll
				for (int i = 0; i < kAhead; i++) a[i] = b[i];
			}
			if (r0 + kManyChunk < rows) stage(buf ^ 1);
			__syncthreads();
		}
	}
	if (e >= E) return;
	const double d = DIRECT ? den[e] : 0.0;
#pragma unroll
	for (int k = 0; k < KT; k++)
		if (k0 + k < K) G[(int64_t)(k0 + k) * E + e] = O::finish(gr[k], gi[k], d, s);
}

// Between the two: a thread per energy and vector, kAhead table rows loaded
// before they are added. There are enough wavefronts to cover the rows' latency
// and not enough for several vectors each.
template <int TYPE, bool DIRECT>
__global__ __launch_bounds__(kThreads) void contract_each(
    const double *__restrict__ L, const double2 *__restrict__ C, const double *__restrict__ den,
    double2 *__restrict__ G, int M, int E, double s) {
	typedef Term<TYPE, DIRECT> O;
	typedef typename O::F F;
	constexpr int kAhead = 16;
	const int e = blockIdx.x * kThreads + threadIdx.x;
	if (e >= E) return;
	const double2 *c = C + (int64_t)blockIdx.y * M;
	double gr = O::start(c[0].x), gi = O::start(c[0].y);
	const int rows = M - O::kFirst;
	c += O::kFirst;
	auto add = [&](F f, double2 cn) __attribute__((always_inline)) {
		const double2 p = O::prepare(cn);
		gr = O::add(f, p, gr);
		gi = O::add(f, O::imag(p), gi);
	};
	int r = 0;
	for (; r + kAhead <= rows; r += kAhead) {
		F f[kAhead];
#pragma unroll
		for (int i = 0; i < kAhead; i++) f[i] = O::load(L, (int64_t)(r + i) * E + e);
#pragma unroll
		for (int i = 0; i < kAhead; i++) add(f[i], c[r + i]);
	}
	for (; r < rows; r++) add(O::load(L, (int64_t)r * E + e), c[r]);
	G[(int64_t)blockIdx.y * E + e] = O::finish(gr, gi, DIRECT ? den[e] : 0.0, s);
}

// Contracts the K vectors in h->gf_in with the array L into h->gf_out.
// contract_many with 8 vectors per wavefront where that gives every SIMD a
// wavefront (4 per CU), with 4 where it gives every CU three; contract_few up to
// one wavefront per SIMD (beyond, some SIMDs run two: 800 energies, 777 moments, 48
// vectors, 1224 wavefronts: 145 us, contract_each 119; 40 vectors, 1020: 105, 109);
// contract_each between. Whole calls at 1000 energies and moments, Retarded, in us:
//   vectors           1    9   37*   64  128  200  256  600   (* 777 x 801)
//   contract_few     67   78  106   206  389  625
//   contract_each    92   98  114   171  288  488  553 1315
//   contract_many                        344  487  544 1324
//   1001 vectors, 2000 moments, 1500 energies: each 6980, many 4050.
template <int TYPE, bool DIRECT>
int contract_launch(tbtkx_context *h, const double *L, const double *den, int K, int M, int E,
                    double s) {
	const double2 *C = h->gf_in.as<double2>();
	double2 *G = h->gf_out.as<double2>();
	const int64_t tiles = (E + 63) / 64, cus = h->num_cus;
	const unsigned grid_x = (unsigned)((E + kThreads - 1) / kThreads);
	auto groups = [&](int kt) { return dim3((unsigned)tiles, (unsigned)((K + 4 * kt - 1) / (4 * kt))); };
	if (tiles * ((K + 7) / 8) >= 4 * cus)
		contract_many<TYPE, DIRECT, 8>
		    <<<groups(8), kThreads, 0, h->stream>>>(L, C, den, G, K, M, E, s);
	else if (tiles * ((K + 3) / 4) >= 3 * cus)
		contract_many<TYPE, DIRECT, 4>
		    <<<groups(4), kThreads, 0, h->stream>>>(L, C, den, G, K, M, E, s);
	else if (((E + 15) / 16) * (int64_t)((K + 1) / 2) <= 4 * cus)
		contract_few<TYPE, DIRECT>
		    <<<dim3((unsigned)((E + 15) / 16), (unsigned)((K + 1) / 2)), 64, 0, h->stream>>>(
		        L, C, den, G, K, M, E, s);
	else
		contract_each<TYPE, DIRECT>
		    <<<dim3(grid_x, (unsigned)K), kThreads, 0, h->stream>>>(L, C, den, G, M, E, s);
	TBTKX_CHECK_HIP(hipGetLastError());
	return TBTKX_OK;
}

template <bool DIRECT>
int contract_type(tbtkx_context *h, int type, const double *L, const double *den, int K, int M,
                  int E, double s) {
	switch (type) {
	case TBTKX_RETARDED: return contract_launch<TBTKX_RETARDED, DIRECT>(h, L, den, K, M, E, s);
	case TBTKX_ADVANCED: return contract_launch<TBTKX_ADVANCED, DIRECT>(h, L, den, K, M, E, s);
	case TBTKX_PRINCIPAL: return contract_launch<TBTKX_PRINCIPAL, DIRECT>(h, L, den, K, M, E, s);
	default: return contract_launch<TBTKX_NONPRINCIPAL, DIRECT>(h, L, den, K, M, E, s);
	}
}

}  // namespace

// Applies the handle's damping (tbtkx_set_damping) to K x M coefficients
// already in device memory, on the handle's stream; no-op without one.
int apply_damping(tbtkx_context *h, double2 *C, int K, int M) {
	if (h->damp_kind == TBTKX_DAMP_NONE || K == 0) return TBTKX_OK;
	if (h->damp_kind == TBTKX_DAMP_LORENTZ && h->damp_broadening == 0) return TBTKX_OK;
	dim3 grid((M + kThreads - 1) / kThreads, K < 1024 ? K : 1024);
	damp_coeffs<<<grid, kThreads, 0, h->stream>>>(C, K, M, h->damp_kind, h->damp_broadening);
	TBTKX_CHECK_HIP(hipGetLastError());
	return TBTKX_OK;
}

// The factors of the direct contraction for one Green's function kind (0:
// e^{-in theta} for Retarded and Advanced, 1: sin(n theta), 2: cos(n theta))
// over n = 1 .. M-1 and the energies e0 + e*de, computed on the host with the
// expressions of generateGreensFunctionCPU (host_math.cpp), so the device
// sums use the reference's values. Kept on the device until another kind,
// order or grid is asked for.
static int direct_factors(tbtkx_context *h, int kind, int M, int E, double e0, double de,
                          double s) {
	if (h->dfac_kind == kind && h->dfac_M == M && h->dfac_E == E && h->dfac_e0 == e0 &&
	    h->dfac_de == de && h->dfac_s == s)
		return TBTKX_OK;
	h->dfac_kind = -1;
	const size_t per = kind == 0 ? 2 : 1;
	const size_t rows = M > 1 ? (size_t)(M - 1) : 0;
	std::vector<double> fac(rows * E * per + per), den(E);
	direct_factor_table(kind, M, E, e0, de, s, fac.data(), den.data());
	int rc;
	if ((rc = h->dfac.reserve(fac.size() * 8))) return rc;
	if ((rc = h->dden.reserve((size_t)E * 8))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->dfac.ptr, fac.data(), fac.size() * 8,
	                               hipMemcpyHostToDevice, h->stream));
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->dden.ptr, den.data(), (size_t)E * 8,
	                               hipMemcpyHostToDevice, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	h->dfac_kind = kind;
	h->dfac_M = M;
	h->dfac_E = E;
	h->dfac_e0 = e0;
	h->dfac_de = de;
	h->dfac_s = s;
	return TBTKX_OK;
}

}  // namespace tbtkx

using namespace tbtkx;

extern "C" {

int tbtkx_lut_upload(tbtkx_handle h, int M, int E, const double *table) {
	TBTKX_REQUIRE(h && table, TBTKX_ERR_ARG, "tbtkx_lut_upload: null pointer");
	TBTKX_LOCK(h);
	TBTKX_REQUIRE(M > 0 && E > 0, TBTKX_ERR_ARG,
	              "tbtkx_lut_upload: table dimensions must be positive");
	int rc = set_device(h);
	if (rc) return rc;
	if ((rc = h->lut.reserve((size_t)M * E * 16))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->lut.ptr, table, (size_t)M * E * 16,
	                               hipMemcpyHostToDevice, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	h->lut_M = M;
	h->lplanes_valid = 0;
	h->lut_E = E;
	return TBTKX_OK;
}

int tbtkx_lut_generate(tbtkx_handle h, int M, int E, double lo, double hi,
                       double s) {
	TBTKX_REQUIRE(h, TBTKX_ERR_ARG, "tbtkx_lut_generate: null handle");
	TBTKX_LOCK(h);
	TBTKX_REQUIRE(M > 0, TBTKX_ERR_ARG,
	              "tbtkx_lut_generate: numCoefficients has to be larger than 0");
	TBTKX_REQUIRE(E > 1, TBTKX_ERR_ARG,
	              "tbtkx_lut_generate: the energy resolution has to be larger than 1");
	TBTKX_REQUIRE(lo < hi, TBTKX_ERR_ARG,
	              "tbtkx_lut_generate: the lower bound has to be smaller than the upper bound");
	TBTKX_REQUIRE(s > 0 && lo > -s && hi < s, TBTKX_ERR_ARG,
	              "tbtkx_lut_generate: the energy window has to lie inside (-s, s)");
	int rc = set_device(h);
	if (rc) return rc;
	if ((rc = h->lut.reserve((size_t)M * E * 16))) return rc;
	const double dx = (hi - lo) / (E - 1);
	dim3 grid((E + kThreads - 1) / kThreads, M);
	lut_generate<<<grid, kThreads, 0, h->stream>>>(h->lut.as<double2>(), M, E,
	                                               lo, dx, s);
	TBTKX_CHECK_HIP(hipGetLastError());
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	h->lut_M = M;
	h->lplanes_valid = 0;
	h->lut_E = E;
	return TBTKX_OK;
}

int tbtkx_lut_destroy(tbtkx_handle h) {
	TBTKX_REQUIRE(h, TBTKX_ERR_ARG, "tbtkx_lut_destroy: null handle");
	TBTKX_LOCK(h);
	int rc = set_device(h);
	if (rc) return rc;
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	h->lut.release();
	h->lut_M = h->lut_E = 0;
	h->lplanes_valid = 0;
	return TBTKX_OK;
}

int tbtkx_set_damping(tbtkx_handle h, int kind, double broadening) {
	TBTKX_REQUIRE(h, TBTKX_ERR_ARG, "tbtkx_set_damping: null handle");
	TBTKX_LOCK(h);
	TBTKX_REQUIRE(kind == TBTKX_DAMP_NONE || kind == TBTKX_DAMP_LORENTZ ||
	                  kind == TBTKX_DAMP_JACKSON,
	              TBTKX_ERR_ARG, "tbtkx_set_damping: unknown damping kind");
	TBTKX_REQUIRE(std::isfinite(broadening), TBTKX_ERR_ARG,
	              "tbtkx_set_damping: the broadening has to be finite");
	h->damp_kind = kind;
	h->damp_broadening = kind == TBTKX_DAMP_LORENTZ ? broadening : 0.0;
	return TBTKX_OK;
}

int tbtkx_contract(tbtkx_handle h, int K, const double *coeffs, int type,
                   double *out) {
	TBTKX_REQUIRE(h, TBTKX_ERR_ARG, "tbtkx_contract: null handle");
	TBTKX_LOCK(h);
	TBTKX_REQUIRE(h->lut_M > 0, TBTKX_ERR_STATE,
	              "tbtkx_contract: no lookup table loaded");
	TBTKX_REQUIRE(K >= 0 && (K == 0 || (coeffs && out)), TBTKX_ERR_ARG,
	              "tbtkx_contract: bad coefficient arrays");
	TBTKX_REQUIRE(type >= TBTKX_ADVANCED && type <= TBTKX_NONPRINCIPAL,
	              TBTKX_ERR_ARG, "tbtkx_contract: unknown Green's function type");
	TBTKX_REQUIRE(K <= 65535, TBTKX_ERR_ARG,
	              "tbtkx_contract: at most 65535 vectors per call");
	if (K == 0) return TBTKX_OK;
	const int M = h->lut_M, E = h->lut_E;
	int rc = set_device(h);
	if (rc) return rc;
	if ((rc = h->gf_in.reserve((size_t)K * M * 16))) return rc;
	if ((rc = h->gf_out.reserve((size_t)K * E * 16))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->gf_in.ptr, coeffs, (size_t)K * M * 16,
	                               hipMemcpyHostToDevice, h->stream));
	if ((rc = apply_damping(h, h->gf_in.as<double2>(), K, M))) return rc;
	if ((rc = contract_type<false>(h, type, h->lut.as<double>(), nullptr, K, M, E, 0.0))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(out, h->gf_out.ptr, (size_t)K * E * 16,
	                               hipMemcpyDeviceToHost, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	return TBTKX_OK;
}

int tbtkx_contract_direct(tbtkx_handle h, int K, int M, const double *coeffs, int type,
                          int E, double e0, double de, double s, double *out) {
	TBTKX_REQUIRE(h, TBTKX_ERR_ARG, "tbtkx_contract_direct: null handle");
	TBTKX_LOCK(h);
	TBTKX_REQUIRE(K >= 0 && K <= 65535 && M > 0 && E > 0 && (K == 0 || (coeffs && out)),
	              TBTKX_ERR_ARG, "tbtkx_contract_direct: bad sizes or arrays");
	TBTKX_REQUIRE(type >= TBTKX_ADVANCED && type <= TBTKX_NONPRINCIPAL, TBTKX_ERR_ARG,
	              "tbtkx_contract_direct: unknown Green's function type");
	TBTKX_REQUIRE(s > 0 && e0 > -s && e0 + (E - 1) * de < s, TBTKX_ERR_ARG,
	              "tbtkx_contract_direct: the energy window has to lie inside (-s, s)");
	if (K == 0) return TBTKX_OK;
	int rc = set_device(h);
	if (rc) return rc;
	if ((rc = h->gf_in.reserve((size_t)K * M * 16))) return rc;
	if ((rc = h->gf_out.reserve((size_t)K * E * 16))) return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(h->gf_in.ptr, coeffs, (size_t)K * M * 16,
	                               hipMemcpyHostToDevice, h->stream));
	if ((rc = apply_damping(h, h->gf_in.as<double2>(), K, M))) return rc;
	const int kind = type == TBTKX_PRINCIPAL ? 1 : type == TBTKX_NONPRINCIPAL ? 2 : 0;
	if ((rc = direct_factors(h, kind, M, E, e0, de, s))) return rc;
	if ((rc = contract_type<true>(h, type, h->dfac.as<double>(), h->dden.as<double>(), K, M, E, s)))
		return rc;
	TBTKX_CHECK_HIP(hipMemcpyAsync(out, h->gf_out.ptr, (size_t)K * E * 16,
	                               hipMemcpyDeviceToHost, h->stream));
	TBTKX_CHECK_HIP(hipStreamSynchronize(h->stream));
	return TBTKX_OK;
}

}  // extern "C"
