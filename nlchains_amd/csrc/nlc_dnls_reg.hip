// DNLS split step of 32 ... 16384-site chains (powers of two) in registers.
//
// Reference behaviour followed: DNLS.cpp:159-175 (as nlc_dnls.hip).
//
// Design: the reference issues 14 cuFFT launches per step, each a full HBM pass
// over the ensemble.  Here N/V threads x V values hold a chain for all steps of
// the batch, V = 8, 16 or 32 (nlc_fft_reg.inl), so HBM is touched once per batch
// (16 B/site in and out).  Two or three passes in registers, where the LDS
// Stockham kernel that ran the lengths up to 2048 made log4 N passes through LDS,
// each with two workgroup barriers, run-time index arithmetic and a table load
// per twiddle.  The Fourier multiplier is read in the order of the spectrum, so
// no reordering pass is ever made.  Up to 1024 sites (2048 with V = 32) a wavefront holds whole chains and never
// waits for another one.
//
// 8192 and 16384 sites are a workgroup's registers (256 and 512 threads x 32
// values, 76 and 139 KB of LDS).
//
// Bound by FP64 issue (about 80 FP64 instructions per point and substep at 1024
// sites) with the LDS exchanges and the twiddle loads beside it.  2^22 sites x
// 20 steps, against the LDS kernel: 32 sites 1.36 ms (3.59), 64 1.50 (3.48),
// 128 1.66 (4.23), 256 1.71 (4.43), 512 1.96 (5.20), 1024 2.15 (6.27), 2048 2.78
// (7.08); one chain of 64 sites 0.20 ms (0.56), of 1024 0.59 (0.95), of 2048
// 0.74 (1.79).  4096 sites x 4096: 9.5 ms against 9.9 with running twiddle powers;
// 8192 x 512 3.09 (7.5) and 16384 x 256 3.57 (7.9) against the two-level form in
// HBM, whose passes are bound by their 64 B per site and substep.
#include "nlc_internal.hpp"

#include <cmath>
#include <type_traits>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"
#include "nlc_fft4096.inl"
#include "nlc_fft_reg.inl"

template <int N, int V>
__global__ void __launch_bounds__((RegFft<N, V>::kBlock), (V == 32 ? 2 : 3))
k_dnls_reg(double2 *__restrict__ state, uint32_t copies, uint32_t steps, DnlsArgs a,
           const double2 *__restrict__ mult) {
	using F = RegFft<N, V>;
	extern __shared__ double lds[]; // F::kLds doubles per chain
	const uint32_t slot = threadIdx.x / F::T, t = threadIdx.x % F::T;
	const uint32_t chain = blockIdx.x * F::kChains + slot;
	const bool live = chain < copies; // a slot past the last chain runs on zeros and writes nothing
	double2 *psi = state + size_t(live ? chain : 0) * N + t;
	double *L = lds + F::kLds * slot;
	double2 v[F::V]; // psi[t + T j] at v[j]
#pragma unroll
	for (int j = 0; j < F::V; ++j) v[j] = live ? psi[F::T * j] : make_double2(0.0, 0.0);
	for (uint32_t s = 0; s < steps; ++s) {
#pragma unroll 1
		for (int k = 0; k < 7; ++k) {
			const double th = (k == 0 && s) ? a.theta[8] : a.theta[k];
			// the twiddles are re-read every substep rather than held in registers
			const double2 *twk = mult + 4 * N;
			asm volatile("" : "+s"(twk));
			nonlinear_groups<V>(v, th);
			reg_fft_fwd<N, V>(v, L, twk, t);
			const double2 *m = mult + size_t(k < 4 ? k : 6 - k) * N + t;
#pragma unroll
			for (int h = 0; h < F::V; h += 8) {
#pragma unroll
				for (int j = h; j < h + 8; ++j) v[j] = cmul(v[j], m[F::T * j]);
				__builtin_amdgcn_sched_barrier(0);
			}
			reg_fft_inv<N, V>(v, L, twk, t);
		}
	}
	if (live) {
#pragma unroll
		for (int j = 0; j < F::V; ++j) psi[F::T * j] = nonlinear(v[j], a.theta[7]);
	}
}

// Row pass of the two-level FFT (nlc_dnls_long.hip) for rows of 4096 points:
// forward FFT, the multipliers T[r + R k] of row r in the spectrum's order, the
// inverse FFT, and the inverse column twiddle W_n^{-m r}; rows[row] in place,
// natural order in and out.  tw: reg_twiddles of 4096 points; twn: the n-point
// roots (n = 4096 R).
__global__ void __launch_bounds__(256, 3)
k_dnls_rows4096(double2 *__restrict__ rows, uint32_t R, const double2 *__restrict__ tw, const double2 *__restrict__ twn,
                const double2 *__restrict__ tk) {
	using F = RegFft<4096, 16>;
	static_assert(F::T == 256, "");
	__shared__ double L[F::kLds];
	const uint32_t row = blockIdx.x, r = row % R, t = threadIdx.x;
	double2 *y = rows + size_t(row) * 4096 + t;
	double2 v[16];
#pragma unroll
	for (int j = 0; j < 16; ++j) v[j] = y[256 * j];
	reg_fft_fwd<4096, 16>(v, L, tw, t);
	const double2 *m = tk + size_t(r) * 4096 + t;
#pragma unroll
	for (int s = 0; s < 16; ++s) v[s] = cmul(v[s], m[256 * s]);
	reg_fft_inv<4096, 16>(v, L, tw, t);
#pragma unroll
	for (int j = 0; j < 16; ++j) y[256 * j] = cmul(v[j], cconj(twn[(t + 256 * j) * r])); // x r < 4096 R = n
}

template <int N, int V>
hipError_t launch_reg(hipStream_t st, double2 *state, uint32_t copies, uint32_t steps, const DnlsArgs &a,
                      const double2 *mult) {
	using F = RegFft<N, V>;
	constexpr size_t lds = sizeof(double) * F::kLds * F::kChains;
	if (lds > 64 * 1024) {
		const hipError_t e = hipFuncSetAttribute((const void *) k_dnls_reg<N, V>, hipFuncAttributeMaxDynamicSharedMemorySize,
		                                         int(lds));
		if (e != hipSuccess) return e;
	}
	hipLaunchKernelGGL((k_dnls_reg<N, V>), dim3((copies + F::kChains - 1) / F::kChains), dim3(F::kBlock), lds, st, state,
	                   copies, steps, a, mult);
	return hipGetLastError();
}

// The 4 multipliers in the order of the spectrum, then the twiddles.
template <int N, int V>
void tables(const double2 *table, double2 *out) {
	using F = RegFft<N, V>;
	for (int k = 0; k < 4; ++k)
		for (uint32_t e = 0; e < N; ++e) out[size_t(k) * N + e] = table[size_t(k) * N + reg_freq<N, V>(e / F::T, e % F::T)];
	out += 4 * N;
	reg_twiddles<N, V>(out);
}

// Values per thread of an ensemble of `copies` chains.  A chain on few threads
// needs fewer exchanges and twiddles per point, one on many finishes sooner, so
// the larger V is taken once its wavefronts fill the 1024 SIMDs (V = 16: at
// 1024 of them, 2^20 sites of 128 550 us against 590; a single chain 401
// against 269) or, at two per SIMD instead of three, one and a half times over
// (V = 32: 1024 sites, 3072 chains 1957 us against 1928 with V = 16, 4096 2147
// against 2519, 1024 1113 against 835; 2048 sites, 1024 chains 1837 against
// 1537, 2048 2855 against 3110).  32 and 64 sites always take V = 8 (2^22 sites
// 1.36 and 1.49 ms against 1.50 with V = 16; 190 against 370 us for one chain).  4096 sites always
// take V = 16 (4096 chains 9.5 ms against 14.5 with V = 32, whose twiddle tables
// and two wavefronts per SIMD do not pay for the smaller exchanges).
int reg_values(uint32_t n, uint32_t copies) {
	const uint64_t sites = uint64_t(n) * copies;
	if (n <= 64) return 8;
	if (n <= 256) return sites >= 1024 * 64 * 16 ? 16 : 8;
	if (n >= 4096) return n == 4096 ? 16 : 32;
	if (sites > 1536 * 64 * 32) return 32;
	return n <= 512 ? 8 : 16;
}

template <int N, int V>
size_t table_size() {
	return 4 * size_t(N) + RegFft<N, V>::kTw;
}

// Calls f<N, V> for the shape of n sites and `copies` chains.
#define NLC_REG_DISPATCH(n, copies, f, ...)                                                                        \
	switch (n * 64 + reg_values(n, copies)) {                                                                       \
	case 32 * 64 + 8: return f<32, 8>(__VA_ARGS__);                                                                 \
	case 64 * 64 + 8: return f<64, 8>(__VA_ARGS__);                                                                 \
	case 128 * 64 + 8: return f<128, 8>(__VA_ARGS__);                                                               \
	case 128 * 64 + 16: return f<128, 16>(__VA_ARGS__);                                                             \
	case 256 * 64 + 8: return f<256, 8>(__VA_ARGS__);                                                               \
	case 256 * 64 + 16: return f<256, 16>(__VA_ARGS__);                                                             \
	case 512 * 64 + 8: return f<512, 8>(__VA_ARGS__);                                                               \
	case 512 * 64 + 32: return f<512, 32>(__VA_ARGS__);                                                             \
	case 1024 * 64 + 16: return f<1024, 16>(__VA_ARGS__);                                                           \
	case 1024 * 64 + 32: return f<1024, 32>(__VA_ARGS__);                                                           \
	case 2048 * 64 + 16: return f<2048, 16>(__VA_ARGS__);                                                           \
	case 2048 * 64 + 32: return f<2048, 32>(__VA_ARGS__);                                                           \
	case 4096 * 64 + 16: return f<4096, 16>(__VA_ARGS__);                                                           \
	case 8192 * 64 + 32: return f<8192, 32>(__VA_ARGS__);                                                           \
	case 16384 * 64 + 32: return f<16384, 32>(__VA_ARGS__);                                                         \
	}

} // namespace

// 8192 and 16384 sites: on chip from 128 chains on; with fewer the rows of the
// two-level form spread over more CUs (20 steps: 8192 sites 1.95 ms for up to 256
// chains against 1.5 for one and 14.7 us for each chain beyond 100; 16384 sites
// 3.2 to 3.6 ms against 1.6 and 31 us).
bool dnls_reg_path(uint32_t n, uint32_t copies) {
	if (n == 8192 || n == 16384) return copies >= 128;
	return n >= 32 && n <= 4096 && (n & (n - 1)) == 0;
}

size_t dnls_reg_table_size(uint32_t n, uint32_t copies) {
	NLC_REG_DISPATCH(n, copies, table_size)
	return 0;
}

void dnls_reg_tables(uint32_t n, uint32_t copies, const double2 *table, double2 *out) {
	NLC_REG_DISPATCH(n, copies, tables, table, out)
}

uint32_t dnls_row4096_freq(uint32_t e) { return reg_freq<4096, 16>(e / 256, e % 256); }
size_t dnls_row4096_twiddles() { return RegFft<4096, 16>::kTw; }
void dnls_row4096_twiddles(double2 *out) { reg_twiddles<4096, 16>(out); }

hipError_t launch_dnls_rows4096(hipStream_t st, double2 *rows, uint32_t nrows, uint32_t R, const double2 *tw,
                                const double2 *twn, const double2 *tk) {
	hipLaunchKernelGGL(k_dnls_rows4096, dim3(nrows), dim3(256), 0, st, rows, R, tw, twn, tk);
	return hipGetLastError();
}

hipError_t launch_dnls_reg(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps,
                           const double *theta9, const double2 *mult) {
	DnlsArgs a;
	for (int i = 0; i < 9; ++i) a.theta[i] = theta9[i];
	NLC_REG_DISPATCH(n, copies, launch_reg, st, state, copies, steps, a, mult)
	return hipErrorInvalidValue;
}

} // namespace nlc
