// DNLS split step of chains up to 4096 sites with a prime factor above 7:
// Bluestein's chirp-z form of the n-point DFTs (L. Bluestein, 1970) on the
// register FFT (nlc_fft_reg.inl).
//
// Reference behaviour followed: DNLS.cpp:159-175 (as nlc_dnls.hip).
//
// With w_j = e^{-i pi j^2/n}, X_k = w_k C_k, C = u * b the cyclic convolution of
// length N >= 2n - 1 (a power of two) of u_x = w_x psi_x with b_j = conj(w_j)
// (|j| < n): conv(u) = IFFT(FFT(u) bhat), bhat = FFT(b)/N.  The chain is kept as
// u_x between substeps, |u_x| = |psi_x|:
//   nonlinear: u_x <- u_x e^{-i theta |u_x|^2};
//   C = conv(u), and the backward DFT of Y = X T as conj(DFT(conj Y)), whose
//   input conj(Y_k) w_k is conj(C_k T_k): u <- conj(conv(conj(C T))).
// The chirps cancel between substeps and are applied only at load and store.
//
// Four N-point transforms per substep, N = 2 to 4 n; half of the values of a
// forward transform are zeros (HALF) and half of those of an inverse one are
// not computed.  Against the LDS form it replaces (radix-4 Stockham passes with
// two barriers each), 20 steps: 11 x 65536 46.8 -> 1.19 ms, 61 x 16384 15.7 ->
// 1.83, 251 x 4096 7.21 -> 2.09, 1021 x 2048 14.0 -> 6.6, 4001 x 256 13.9 -> 7.5;
// one chain of 101 sites 0.85 -> 0.52 ms.
#include "nlc_internal.hpp"

#include <cmath>
#include <type_traits>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"
#include "nlc_fft4096.inl"
#include "nlc_fft_reg.inl"

// table: bhat in the spectrum's order (N), the twiddles (kTw), the 4 distinct
// multipliers (4 n), the chirp (n).
template <int N, int V>
__global__ void __launch_bounds__((RegFft<N, V>::kBlock), (V == 32 ? 2 : 3))
k_dnls_blue(double2 *__restrict__ state, uint32_t n, uint32_t copies, uint32_t steps, DnlsArgs a,
            const double2 *__restrict__ table) {
	using F = RegFft<N, V>;
	constexpr uint32_t T = F::T;
	constexpr int H = V / 2; // values of the chain per thread: n <= N/2
	extern __shared__ double lds[]; // F::kLds doubles per chain
	const uint32_t slot = threadIdx.x / T, t = threadIdx.x % T;
	const uint32_t chain = blockIdx.x * F::kChains + slot;
	const bool live = chain < copies; // a slot past the last chain runs on zeros and writes nothing
	double2 *psi = state + size_t(live ? chain : 0) * n + t;
	double *L = lds + F::kLds * slot;
	const double2 *mult = table + N + F::kTw, *chirp = mult + size_t(4) * n + t;
	const double2 zero = make_double2(0.0, 0.0);
	double2 v[V];
#pragma unroll
	for (int j = 0; j < H; ++j) v[j] = live && t + T * j < n ? cmul(psi[T * j], chirp[T * j]) : zero;
	// v <- conv(v) on the first half, the tables re-read rather than held in registers
	const auto conv = [&] {
		const double2 *tab = table;
		asm volatile("" : "+s"(tab));
		reg_fft_fwd<N, V, true>(v, L, tab + N, t);
#pragma unroll
		for (int h = 0; h < V; h += 8) {
#pragma unroll
			for (int s = h; s < h + 8; ++s) v[s] = cmul(v[s], tab[T * s + t]);
			__builtin_amdgcn_sched_barrier(0);
		}
		reg_fft_inv<N, V>(v, L, tab + N, t);
	};
	for (uint32_t s = 0; s < steps; ++s) {
#pragma unroll 1
		for (int k = 0; k < 7; ++k) {
			const double th = (k == 0 && s) ? a.theta[8] : a.theta[k];
			nonlinear_groups<H>(v, th);
			const double2 *tk = mult + size_t(k < 4 ? k : 6 - k) * n + t;
#pragma unroll 1
			for (int half = 0; half < 2; ++half) {
				conv();
				// conj(C T), then conj of the second convolution; zero past the chain
				if (half == 0) {
#pragma unroll
					for (int g = 0; g < H; g += 4) {
#pragma unroll
						for (int j = g; j < g + 4; ++j) v[j] = t + T * j < n ? cconj(cmul(v[j], tk[T * j])) : zero;
						__builtin_amdgcn_sched_barrier(0);
					}
				} else {
#pragma unroll
					for (int j = 0; j < H; ++j) v[j] = t + T * j < n ? cconj(v[j]) : zero;
				}
			}
		}
	}
	if (live) {
#pragma unroll
		for (int j = 0; j < H; ++j)
			if (t + T * j < n) psi[T * j] = nonlinear(cmul(v[j], cconj(chirp[T * j])), a.theta[7]);
	}
}

template <int N, int V>
hipError_t launch_blue(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps, const DnlsArgs &a,
                       const double2 *table) {
	using F = RegFft<N, V>;
	constexpr size_t lds = sizeof(double) * F::kLds * F::kChains;
	if (lds > 64 * 1024) {
		const hipError_t e = hipFuncSetAttribute((const void *) k_dnls_blue<N, V>,
		                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
		if (e != hipSuccess) return e;
	}
	hipLaunchKernelGGL((k_dnls_blue<N, V>), dim3((copies + F::kChains - 1) / F::kChains), dim3(F::kBlock), lds, st, state,
	                   n, copies, steps, a, table);
	return hipGetLastError();
}

template <int N, int V>
size_t table_size(uint32_t n) {
	return N + RegFft<N, V>::kTw + size_t(5) * n;
}

template <int N, int V>
void tables(uint32_t n, const double2 *mult, const double2 *blue, double2 *out) {
	using F = RegFft<N, V>; // blue: bhat, roots, chirp
	for (uint32_t e = 0; e < uint32_t(N); ++e) out[e] = blue[reg_freq<N, V>(e / F::T, e % F::T)];
	reg_twiddles<N, V>(out + N);
	out += N + F::kTw;
	std::copy(mult, mult + size_t(4) * n, out);
	std::copy(blue + 2 * size_t(N), blue + 2 * size_t(N) + n, out + size_t(4) * n);
}

// Values per thread: as the power-of-two kernels (nlc_dnls_reg.hip), by the
// sites of the convolutions.
int blue_values(uint32_t N, uint32_t copies) {
	const uint64_t sites = uint64_t(N) * copies;
	if (N <= 64) return 8;
	if (N <= 256) return sites >= 1024 * 64 * 16 ? 16 : 8;
	if (N == 8192 || (N <= 2048 && sites > 1536 * 64 * 32)) return 32;
	return N <= 512 ? 8 : 16;
}

#define NLC_BLUE_DISPATCH(n, copies, f, ...)                                                                       \
	switch (const uint32_t N_ = dnls_bluestein_size(n); N_ * 64 + blue_values(N_, copies)) {                        \
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
	}

} // namespace

size_t dnls_blue_table_size(uint32_t n, uint32_t copies) {
	NLC_BLUE_DISPATCH(n, copies, table_size, n)
	return 0;
}

void dnls_blue_tables(uint32_t n, uint32_t copies, const double2 *mult, const double2 *blue, double2 *out) {
	NLC_BLUE_DISPATCH(n, copies, tables, n, mult, blue, out)
}

hipError_t launch_dnls_blue(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps,
                            const double *theta9, const double2 *table) {
	DnlsArgs a;
	for (int i = 0; i < 9; ++i) a.theta[i] = theta9[i];
	NLC_BLUE_DISPATCH(n, copies, launch_blue, st, state, n, copies, steps, a, table)
	return hipErrorInvalidValue;
}

} // namespace nlc
