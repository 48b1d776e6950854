// DNLS split step of chains up to 8192 sites whose prime factors are 2, 3, 5
// and 7 (3000, 5000, 6000, ...; the powers of two from 32 on have their own
// kernels), chain resident in LDS for a whole batch.
//
// Reference behaviour followed: DNLS.cpp:159-175 (as nlc_dnls.hip).
//
// Design: the in-place passes of nlc_smooth_plan.inl.  The butterflies of the
// first forward and the last inverse pass are the same elements, and with the
// nonlinear phase between them they make one sweep over the chain (outer), as
// the last forward pass, the Fourier multiplier and the first inverse pass do
// (inner): 2 m - 2 sweeps per substep for m passes, each reading and writing the
// chain once in LDS with one workgroup barrier.  Twiddles and multipliers are
// tables in the order of use.
//
// Bound by latency: LDS round trip, twiddle loads from L2 and a barrier per
// sweep, with the 9 to 12 wavefronts per CU that the chains' LDS leaves; FP64
// issue is about half of the time.  Against radix 2, 3, 4, 5 and 7 Stockham passes
// (two barriers each, run-time divisions, direct sums), 20 steps: 1000 x 2048
// 5.80 -> 1.98 ms, 500 x 4096 4.10 -> 1.91, 100 x 20000 3.31 -> 1.22, 3000 x 1024
// 7.9 -> 3.8, 5000 x 512 6.5 -> 2.8, 30 x 65536 2.96 -> 1.32; one chain of 1000
// sites 1.57 -> 0.98; 12 x 200000 (a thread per chain) 2.93 -> 0.58.
#include "nlc_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"
#include "nlc_fft4096.inl"
#include "nlc_fft_reg.inl"
#include "nlc_fft_smooth.inl"

#include "nlc_smooth_plan.inl"

// last inverse pass, nonlinear phase, first forward pass
template <int P>
__device__ __forceinline__ void outer(const SmoothCtx &cx, const SmoothPass &ps, double theta, bool inverse,
                                      bool forward) {
	for_butterflies<P, false>(cx, ps, [&](double2 *a, uint32_t, uint32_t rest) {
		const double2 *w = cx.tw + ps.tw + rest;
		if (inverse) {
			twiddle_conj<P>(a, w, ps.per_block.d);
			dft_nat<P, +1>(a);
		}
		nonlinear_groups<P>(a, theta);
		if (forward) {
			asm volatile("" : "+v"(w)); // read the twiddles again rather than hold them over the nonlinear phase
			then_multiply<P, 1>(a, w, ps.per_block.d, [](double2 *v) { dft_nat<P, -1>(v); });
		}
	});
}

// last forward pass, Fourier multiplier ([k][j], the order of the sweep), first inverse pass
template <int P>
__device__ __forceinline__ void inner(const SmoothCtx &cx, const SmoothPass &ps, const double2 *__restrict__ mult) {
	for_butterflies<P, true>(cx, ps, [&](double2 *a, uint32_t j, uint32_t) {
		then_multiply<P, 0>(a, mult + j, ps.nb, [](double2 *v) { dft_nat<P, -1>(v); });
		dft_nat<P, +1>(a);
	});
}

// table: the plan (kPlanValues), 4 multipliers of n values, the twiddles.
// Registers: 128 for MAXP = 10, the plans without a larger radix (1000 x 2048
// 2.10 ms with the other kernel, 1.98 with this; 5000 x 512 3.37 and 2.80); 178 for 16,
// which at three waves per SIMD spilled 15 of them (1200 x 2048 2.80 ms, at two
// 2.47; 8100 x 300 7.17 and 5.24).
template <int MAXP>
__global__ void __launch_bounds__(kMaxBlock, MAXP <= 10 ? 3 : 2)
k_dnls_smooth(double2 *__restrict__ state, uint32_t copies, uint32_t chains, uint32_t steps, DnlsArgs a,
              const double2 *__restrict__ table) {
	extern __shared__ double2 buf[];
	const SmoothPlan *plan = reinterpret_cast<const SmoothPlan *>(table);
	const uint32_t n = plan->n, m = plan->m, first = blockIdx.x * chains;
	const double2 *mult = table + kPlanValues;
	const SmoothCtx cx{buf, chains, plan->lds_chain, plan->pad, plan->last, mult + size_t(4) * n};
	const uint32_t live = min(chains, copies - first); // chains past the last one run on zeros
	double2 *psi = state + size_t(first) * n;
	for (uint32_t c = 0; c < chains; ++c)
		for (uint32_t e = threadIdx.x; e < n; e += blockDim.x)
			buf[c * cx.lds_chain + e + cx.pad * cx.last.div(e)] = c < live ? psi[size_t(c) * n + e] : make_double2(0.0, 0.0);
	__syncthreads();
	for (uint32_t s = 0; s < steps; ++s) {
		for (int k = 0; k < 7; ++k) {
			const double th = (k == 0 && s) ? a.theta[8] : a.theta[k];
			const bool inverse = s || k;
			const SmoothPass p0 = plan->p[0];
#define NLC_F(P) outer<P>(cx, p0, th, inverse, true)
			NLC_RADIX_SWITCH(MAXP, p0.radix, NLC_F)
#undef NLC_F
			__syncthreads();
			for (uint32_t i = 1; i + 1 < m; ++i) {
				const SmoothPass pi = plan->p[i];
#define NLC_F(P) middle<P, false>(cx, pi)
				NLC_RADIX_SWITCH(MAXP, pi.radix, NLC_F)
#undef NLC_F
				__syncthreads();
			}
			const SmoothPass pl = plan->p[m - 1];
			const double2 *mk = mult + size_t(k < 4 ? k : 6 - k) * n;
#define NLC_F(P) inner<P>(cx, pl, mk)
			NLC_RADIX_SWITCH(MAXP, pl.radix, NLC_F)
#undef NLC_F
			__syncthreads();
			for (uint32_t i = m - 1; i-- > 1;) {
				const SmoothPass pi = plan->p[i];
#define NLC_F(P) middle<P, true>(cx, pi)
				NLC_RADIX_SWITCH(MAXP, pi.radix, NLC_F)
#undef NLC_F
				__syncthreads();
			}
		}
	}
	const SmoothPass p0 = plan->p[0];
#define NLC_F(P) outer<P>(cx, p0, a.theta[7], true, false)
	NLC_RADIX_SWITCH(MAXP, p0.radix, NLC_F)
#undef NLC_F
	__syncthreads();
	for (uint32_t c = 0; c < live; ++c)
		for (uint32_t e = threadIdx.x; e < n; e += blockDim.x)
			psi[size_t(c) * n + e] = buf[c * cx.lds_chain + e + cx.pad * cx.last.div(e)];
}

// Chains of n = 2 ... 16 sites: a thread per chain, one butterfly per transform.
// table: the 4 multipliers, natural order.
template <int P>
__global__ void __launch_bounds__(64)
k_dnls_tiny(double2 *__restrict__ state, uint32_t copies, uint32_t steps, DnlsArgs a, const double2 *__restrict__ mult) {
	const uint32_t chain = blockIdx.x * 64 + threadIdx.x;
	if (chain >= copies) return;
	double2 *psi = state + size_t(chain) * P;
	double2 v[P];
#pragma unroll
	for (int j = 0; j < P; ++j) v[j] = psi[j];
	for (uint32_t s = 0; s < steps; ++s) {
#pragma unroll 1
		for (int k = 0; k < 7; ++k) {
			nonlinear_groups<P>(v, (k == 0 && s) ? a.theta[8] : a.theta[k]);
			dft_nat<P, -1>(v);
			const double2 *m = mult + (k < 4 ? k : 6 - k) * P;
#pragma unroll
			for (int j = 0; j < P; ++j) v[j] = cmul(v[j], m[j]);
			dft_nat<P, +1>(v);
		}
	}
#pragma unroll
	for (int j = 0; j < P; ++j) psi[j] = nonlinear(v[j], a.theta[7]);
}

bool radices_to_10(const SmoothPlan &pl) {
	for (uint32_t i = 0; i < pl.m; ++i)
		if (pl.p[i].radix > 10) return false;
	return true;
}

} // namespace

bool dnls_smooth_path(uint32_t n) {
	return smooth_length(n) || n == 2 || n == 4 || n == 8 || n == 16;
}

size_t dnls_smooth_table_size(uint32_t n) {
	if (n <= 16) return size_t(4) * n;
	const SmoothPlan pl = make_plan(n);
	return kPlanValues + size_t(4) * n + smooth_twiddles(pl);
}

void dnls_smooth_tables(uint32_t n, const double2 *table, double2 *out) {
	if (n <= 16) {
		std::copy(table, table + size_t(4) * n, out);
		return;
	}
	const SmoothPlan pl = make_plan(n);
	std::memcpy((void *) out, &pl, sizeof pl);
	out += kPlanValues;
	const SmoothPass &in = pl.p[pl.m - 1];
	for (uint32_t e = 0; e < n; ++e) {
		const uint32_t f = smooth_freq(pl, e);
		const uint32_t at = (e % in.radix) * in.nb + e / in.radix;
		for (int k = 0; k < 4; ++k) out[size_t(k) * n + at] = table[size_t(k) * n + f];
	}
	out += size_t(4) * n;
	smooth_fill_twiddles(pl, out);
}

hipError_t launch_dnls_smooth(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps,
                              const double *theta9, const double2 *table) {
	DnlsArgs a;
	for (int i = 0; i < 9; ++i) a.theta[i] = theta9[i];
	if (n <= 16) {
#define NLC_F(P)                                                                                                   \
	hipLaunchKernelGGL(k_dnls_tiny<P>, dim3((copies + 63) / 64), dim3(64), 0, st, state, copies, steps, a, table)
		NLC_RADIX_SWITCH(16, n, NLC_F)
#undef NLC_F
		return hipGetLastError();
	}
	const SmoothPlan plan = make_plan(n);
	uint32_t chains = 1;
	const uint32_t block = choose_block(plan, copies, chains);
	const size_t lds = sizeof(double2) * plan.lds_chain * chains;
	const auto kernel = radices_to_10(plan) ? k_dnls_smooth<10> : k_dnls_smooth<16>;
	if (lds > 64 * 1024) {
		const hipError_t e = hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
		                                         int(lds));
		if (e != hipSuccess) return e;
	}
	hipLaunchKernelGGL(kernel, dim3((copies + chains - 1) / chains), dim3(block), lds, st, state, copies, chains,
	                   steps, a, table);
	return hipGetLastError();
}

} // namespace nlc
