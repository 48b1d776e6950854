// DNLS split-step Yoshida-6 integrator, chain resident on chip for a whole batch.
//
// Reference behaviour followed: DNLS.cpp:159-175 (per substep k: nonlinear
// rotation by beta dt c_k with the merged 2 c_0, forward FFT, Fourier multiplier
// T_k = exp(-i dt d_k w)/N (DNLS/dispersion.cpp:19-26), inverse FFT; a final
// beta dt c_7 rotation after the batch), kernels DNLS.cu:11-25 and the cuFFT
// load callbacks DNLS.cu:45-67; CPU form DNLS/cpu-implementation/DNLS.cpp:110-128.
//
// This file: the choice of the kernel for a chain length, and the radix-8 kernel
// of 4096-site chains (k_dnls_4096_r8).  The other kernels: nlc_dnls_reg.hip
// (powers of two in registers), nlc_dnls_smooth.hip (prime factors 2, 3, 5, 7),
// nlc_dnls_blue.hip (other lengths up to 4096) and nlc_dnls_long.hip (the longer
// ones, in HBM).
#include "nlc_internal.hpp"
#include "nlc_fft_large.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"

// ---------------------------------------------------------------- radix 16

#include "nlc_fft4096.inl"
#include "nlc_fft_reg.inl"


// ---------------------------------------------------------------- radix 8
//
// k_dnls_4096_r8: 512 threads x 8 complex values, 4096 = 8^4 in four radix-8
// passes.  Same DFT and twiddle work per point as the radix-16 kernel, half
// the values per thread, so about half the VGPRs and twice the wavefronts per
// SIMD to hide L2 and LDS latency, for one more LDS exchange per transform.
// Digits: x = x0 + 8 x1 + 64 x2 + 512 x3, k = k0 + 8 k1 + 64 k2 + 512 k3;
// thread t = lane + 64 w.

constexpr int kT8 = 512;

// v[at(j)] *= W^{e0 + j de}, j = 0..7, W = exp(-2 pi i/4096) = tw[1] (conjugated
// when CONJ), at(j) = pos8(j) when TRANSPOSED; powers refreshed from the table
// at j = 0 and 4.  ONE0 asserts e0 == 0.
template <bool CONJ, bool ONE0, bool TRANSPOSED>
__device__ __forceinline__ void twiddle_run8(double2 v[8], const double2 *__restrict__ tw, uint32_t e0, uint32_t de) {
	const double2 w = tw[de & 4095u];
	const double2 wc = CONJ ? cconj(w) : w;
#pragma unroll
	for (int q = 0; q < 2; ++q) {
		double2 r = tw[(e0 + uint32_t(4 * q) * de) & 4095u];
		if (CONJ) r = cconj(r);
#pragma unroll
		for (int j = 0; j < 4; ++j) {
			const int idx = 4 * q + j;
			const int at = TRANSPOSED ? pos8(idx) : idx;
			if (idx || !ONE0) v[at] = cmul(v[at], r);
			if (j < 3) r = cmul(r, wc);
		}
	}
}

// LDS layout of the radix-8 kernel: wavefront w owns the 640 entries from
// kR8Region w (dynamic LDS, 8 x 640 x 16 B = 80 KB per chain, two chains per
// CU).  The cross-wave exchange puts element (t, k0) at kR8Region k0 + t, so
// the wavefront w = k0 that gathers it reads only its own region; the two
// in-wave exchanges are 8 x 8 transposes per group of 8 lanes through padded
// rows (stride 9) inside the same region.  Every slot is a per-lane base plus
// a compile-time offset (no per-register address arithmetic), and 16
// consecutive lanes touch distinct bank quads except for one pair in the
// read of exchange 2.
//   exchange 2: element (x0, x1, k1) at 9 (x0 + 8 x1) + k1, written by lane
//               x0 + 8 x1 (offset k1), read by lane x0 + 8 k1 (offset 72 x1)
//   exchange 3: element (x0, k1, k2) at 72 k1 + 9 x0 + k2, written by lane
//               x0 + 8 k1 (offset k2), read by lane k2 + 8 k1 (offset 9 x0)
constexpr uint32_t kR8Region = 640;
constexpr uint32_t kR8Lds = 8 * kR8Region * sizeof(double2);

// Forward FFT.  In: thread t holds psi[t + 512 x3] at v[pos8(x3)].  Out: thread
// t = k2 + 8 k1 + 64 k0 holds X[k0 + 8 k1 + 64 k2 + 512 k3] at v[pos8(k3)].
// LDS hazards as in fft4096_fwd: exchange 1 writes only slots the same thread
// read last, every other write lands in the wavefront's own region.
__device__ __forceinline__ void fft4096_fwd8(double2 v[8], double2 *L, const double2 *__restrict__ tw) {
	const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6, lo = lane & 7, hi = lane >> 3;
	double2 *own = L + kR8Region * w;
	// A: over x3 -> k0 (natural), twiddle W^{t k0}
	dft8_t2n<-1>(v);
	twiddle_run8<false, true, false>(v, tw, 0, t);
	// exchange 1 (cross-wave); thread (lane, w = k0) gathers x2
	double2 *x1w = L + t;
#pragma unroll
	for (int k0 = 0; k0 < 8; ++k0) x1w[kR8Region * k0] = v[k0];
	lds_barrier();
	const double2 *x1r = own + lane;
#pragma unroll
	for (int x2 = 0; x2 < 8; ++x2) v[x2] = x1r[64 * x2];
	// B: over x2 -> k1 (transposed), twiddle W^{8 (x0 + 8 x1) k1}, x0 + 8 x1 = lane
	dft8_n2t<-1>(v);
	twiddle_run8<false, true, true>(v, tw, 0, 8 * lane);
	// exchange 2 (in-wave): lane (x0 = lo, x1 = hi) -> lane (x0 = lo, k1 = hi)
	wave_sync();
	double2 *x2w = own + 9 * lane;
#pragma unroll
	for (int k1 = 0; k1 < 8; ++k1) x2w[k1] = v[pos8(k1)];
	wave_sync();
	const double2 *x2r = own + 9 * lo + hi;
#pragma unroll
	for (int x1 = 0; x1 < 8; ++x1) v[x1] = x2r[72 * x1];
	// C: over x1 -> k2 (transposed), twiddle W^{64 x0 k2}
	dft8_n2t<-1>(v);
	twiddle_run8<false, true, true>(v, tw, 0, 64 * lo);
	// exchange 3 (in-wave): lane (x0 = lo, k1 = hi) -> lane (k2 = lo, k1 = hi)
	wave_sync();
	double2 *x3w = own + 72 * hi + 9 * lo;
#pragma unroll
	for (int k2 = 0; k2 < 8; ++k2) x3w[k2] = v[pos8(k2)];
	wave_sync();
	const double2 *x3r = own + 72 * hi + lo;
#pragma unroll
	for (int x0 = 0; x0 < 8; ++x0) v[x0] = x3r[9 * x0];
	// D: over x0 -> k3 (transposed)
	dft8_n2t<-1>(v);
}

// Inverse (unnormalised) FFT, the exact reverse of fft4096_fwd8.
__device__ __forceinline__ void fft4096_inv8(double2 v[8], double2 *L, const double2 *__restrict__ tw) {
	const uint32_t t = threadIdx.x, lane = t & 63, w = t >> 6, lo = lane & 7, hi = lane >> 3;
	double2 *own = L + kR8Region * w;
	// D': over k3 -> x0 (natural), twiddle W^{-64 x0 k2}, k2 = lo
	dft8_t2n<+1>(v);
	twiddle_run8<true, true, false>(v, tw, 0, 64 * lo);
	// exchange 3': lane (k2 = lo, k1 = hi) -> lane (x0 = lo, k1 = hi)
	wave_sync();
	double2 *x3w = own + 72 * hi + lo;
#pragma unroll
	for (int x0 = 0; x0 < 8; ++x0) x3w[9 * x0] = v[x0];
	wave_sync();
	const double2 *x3r = own + 72 * hi + 9 * lo;
#pragma unroll
	for (int k2 = 0; k2 < 8; ++k2) v[pos8(k2)] = x3r[k2];
	// C': over k2 -> x1 (natural), twiddle W^{-8 (x0 + 8 x1) k1}, x0 = lo, k1 = hi
	dft8_t2n<+1>(v);
	twiddle_run8<true, false, false>(v, tw, 8 * lo * hi, 64 * hi);
	// exchange 2': lane (x0 = lo, k1 = hi) -> lane (x0 = lo, x1 = hi)
	wave_sync();
	double2 *x2w = own + 9 * lo + hi;
#pragma unroll
	for (int x1 = 0; x1 < 8; ++x1) x2w[72 * x1] = v[x1];
	wave_sync();
	const double2 *x2r = own + 9 * lane;
#pragma unroll
	for (int k1 = 0; k1 < 8; ++k1) v[pos8(k1)] = x2r[k1];
	// B': over k1 -> x2 (natural), twiddle W^{-(lane + 64 x2) k0}, k0 = w
	dft8_t2n<+1>(v);
	twiddle_run8<true, false, false>(v, tw, lane * w, 64 * w);
	// exchange 1' (cross-wave), written into the wavefront's own region
	wave_sync();
	double2 *x1w = own + lane;
#pragma unroll
	for (int x2 = 0; x2 < 8; ++x2) x1w[64 * x2] = v[x2];
	lds_barrier();
	const double2 *x1r = L + t;
#pragma unroll
	for (int k0 = 0; k0 < 8; ++k0) v[k0] = x1r[kR8Region * k0];
	// A': over k0 -> x3 (transposed)
	dft8_n2t<+1>(v);
}

__global__ void __launch_bounds__(kT8, 4)
k_dnls_4096_r8(double2 *__restrict__ state, uint32_t copies, uint32_t steps, DnlsArgs a,
               const double2 *__restrict__ tw, const double2 *__restrict__ mult) {
	extern __shared__ double2 lds8[]; // kR8Lds bytes
	const uint32_t chain = blockIdx.x, t = threadIdx.x;
	double2 *psi = state + size_t(chain) * 4096;
	double2 v[8]; // psi[t + 512 j] at v[pos8(j)]
#pragma unroll
	for (int j = 0; j < 8; ++j) v[pos8(j)] = psi[t + 512 * j];
	for (uint32_t s = 0; s < steps; ++s) {
#pragma unroll 1
		for (int k = 0; k < 7; ++k) {
			const double th = (k == 0 && s) ? a.theta[8] : a.theta[k];
			const double2 *twk = tw;
			asm volatile("" : "+s"(twk));
			nonlinear_all(v, th);
			fft4096_fwd8(v, lds8, twk);
			// Fourier multiplier, stored per thread in the digit-reversed order;
			// the fence keeps its loads out of the transform (4 wavefronts per
			// SIMD hide their latency, registers are the scarce resource here)
			asm volatile("" ::: "memory");
			const double2 *m = mult + size_t(k < 4 ? k : 6 - k) * 4096 + t;
#pragma unroll
			for (int j = 0; j < 8; ++j) v[pos8(j)] = cmul(v[pos8(j)], m[512 * j]);
			fft4096_inv8(v, lds8, twk);
		}
	}
#pragma unroll
	for (int j = 0; j < 8; ++j) psi[t + 512 * j] = nonlinear(v[pos8(j)], a.theta[7]);
}

} // namespace

bool dnls_supported(uint32_t n) {
	uint32_t R, M;
	return dnls_reg_path(n, 1) || dnls_smooth_path(n) || dnls_bluestein_size(n) != 0 ||
	       dnls_two_level(n) || large_fft_split(n, R, M) || bluestein_two_level_size(n) != 0;
}

// The 4 distinct Fourier multipliers (d_k = d_{6-k}) in the order the radix-8
// kernel reads them: entry [k][512 j + t] = T_k[(t >> 6) + 8 ((t >> 3) & 7) + 64 (t & 7) + 512 j].
bool dnls_fast_path(uint32_t n) { return n == 4096; }

void dnls_radix8_tables(const double2 *table, double2 *out) {
	for (int k = 0; k < 4; ++k)
		for (uint32_t e = 0; e < 4096; ++e) {
			const uint32_t j = e >> 9, t = e & 511;
			out[size_t(k) * 4096 + e] = table[size_t(k) * 4096 + (t >> 6) + 8 * ((t >> 3) & 7) + 64 * (t & 7) + 512 * j];
		}
}

hipError_t launch_dnls(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps,
                       const double *theta9, const double2 *tw, const double2 *table, int variant, double2 *scratch,
                       const double2 *blue) {
	if (variant == kDnlsRadix8 && dnls_fast_path(n)) {
		DnlsArgs a;
		for (int i = 0; i < 9; ++i) a.theta[i] = theta9[i];
		const hipError_t e = hipFuncSetAttribute((const void *) k_dnls_4096_r8, hipFuncAttributeMaxDynamicSharedMemorySize,
		                                         int(kR8Lds));
		if (e != hipSuccess) return e;
		hipLaunchKernelGGL(k_dnls_4096_r8, dim3(copies), dim3(kT8), kR8Lds, st, state, copies, steps, a, tw, table);
		return hipGetLastError();
	}
	if (dnls_reg_path(n, copies)) return launch_dnls_reg(st, state, n, copies, steps, theta9, table);
	if (dnls_smooth_path(n)) return launch_dnls_smooth(st, state, n, copies, steps, theta9, table);
	if (dnls_bluestein_size(n)) return launch_dnls_blue(st, state, n, copies, steps, theta9, table);
	return launch_dnls_long(st, state, n, copies, steps, theta9, tw, table, scratch, blue);
}

} // namespace nlc
