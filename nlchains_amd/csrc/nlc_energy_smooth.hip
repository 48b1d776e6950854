// Linear-mode energy pass of chains up to 8192 sites whose prime factors are 2,
// 3, 5 and 7 (the powers of two from 8 on have their own kernels).  Reference
// behaviour and formulas as nlc_energy.hip.
//
// Design: several chains per workgroup in LDS, transformed by the in-place
// sweeps of nlc_smooth_plan.inl; mode k of a chain is read from the place of Z_k
// (and of Z_{n-k}, real models) through a table of places, and each thread
// accumulates its modes over the chains in registers.  Up to 16 sites a thread
// transforms a whole chain in registers.
//
// Bound by the latency of the sweeps, as the DNLS kernel; the state is read once.
// Whole pass at 4.2 million sites (67 MB), against one chain per workgroup with
// radix 2, 3, 4, 5 and 7 Stockham passes: 20 sites 72 us (1154), 48 60 (618), 100 63
// (355), 360 70 (173), 1000 89 (105), 5000 98 (167), 7000 116 (167); 12 x 300000 32
// us (1658).
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

// |P - i w Q|^2 of z = q + i p from Z_k and Z_{n-k}, times 4 (see nlc_energy.hip)
__device__ __forceinline__ double mode_energy4(double2 z, double2 zm, double w) {
	const double a = 1.0 + w, b = 1.0 - w;
	const double er = fma(a, z.x, -b * zm.x), ei = fma(a, z.y, b * zm.y);
	return fma(er, er, ei * ei);
}

constexpr int kModes = 16; // modes per thread: n <= 16 blockDim.x

// table: the plan (kPlanValues), the twiddles (ntw), then for every mode the
// places of Z_k (low half) and Z_{n-k} in LDS, 4 modes to a value.
// Two waves per SIMD with both spectra's values (211 registers; at three 44
// spilled: 1000 x 4096 89 -> 65 us, 5000 x 1024 103 -> 80), three with one (1200 x
// 4096 70 us, at two 82).
template <bool DNLS_MODE>
__global__ void __launch_bounds__(kMaxBlock, DNLS_MODE ? 3 : 2)
k_energy_smooth(const double2 *__restrict__ state, uint32_t copies, uint32_t chains, uint32_t ntw,
                const double2 *__restrict__ table, const double *__restrict__ omega, double *__restrict__ partial) {
	extern __shared__ double2 buf[];
	const SmoothPlan *plan = reinterpret_cast<const SmoothPlan *>(table);
	const uint32_t n = plan->n, m = plan->m;
	const SmoothCtx cx{buf, chains, plan->lds_chain, plan->pad, plan->last, table + kPlanValues};
	const uint32_t *places = reinterpret_cast<const uint32_t *>(table + kPlanValues + ntw);
	// n <= blockDim.x: the threads form groups that share the chains of a round
	const uint32_t groups = max(1u, blockDim.x / n), group = n <= blockDim.x ? threadIdx.x / n : 0;
	const uint32_t k0 = threadIdx.x - group * n;
	double acc[kModes];
#pragma unroll
	for (int i = 0; i < kModes; ++i) acc[i] = 0.0;
	for (uint32_t first = blockIdx.x * chains; first < copies; first += gridDim.x * chains) {
		const uint32_t live = min(chains, copies - first);
		const double2 *z = state + size_t(first) * n;
		for (uint32_t c = 0; c < live; ++c)
			for (uint32_t e = threadIdx.x; e < n; e += blockDim.x)
				buf[c * cx.lds_chain + e + cx.pad * cx.last.div(e)] = z[size_t(c) * n + e];
		__syncthreads();
		// chains past the last one are transformed too (whatever they hold) and not read
		for (uint32_t i = 0; i < m; ++i) {
			const SmoothPass ps = plan->p[i];
			if (i + 1 < m) {
#define NLC_F(P) middle<P, false>(cx, ps)
				NLC_RADIX_SWITCH(16, ps.radix, NLC_F)
#undef NLC_F
			} else {
#define NLC_F(P) for_butterflies<P, true>(cx, ps, [](double2 *a, uint32_t, uint32_t) { dft_nat<P, -1>(a); })
				NLC_RADIX_SWITCH(16, ps.radix, NLC_F)
#undef NLC_F
			}
			__syncthreads();
		}
		if (group < groups) {
#pragma unroll
			for (int i = 0; i < kModes; ++i) {
				const uint32_t k = k0 + i * blockDim.x;
				if (k >= n) break;
				const uint32_t at = places[k];
				const double w = DNLS_MODE ? 0.0 : omega[k];
				for (uint32_t c = group; c < live; c += groups) {
					const double2 *x = buf + c * cx.lds_chain;
					const double2 v = x[at & 0xffff];
					if constexpr (DNLS_MODE) acc[i] += fma(v.x, v.x, v.y * v.y);
					else acc[i] += mode_energy4(v, x[at >> 16], w);
				}
			}
		}
		__syncthreads();
	}
	const double scale = DNLS_MODE ? 1.0 : 0.25;
	double *row = partial + size_t(blockIdx.x) * n;
	if (n > blockDim.x) {
#pragma unroll
		for (int i = 0; i < kModes; ++i) {
			const uint32_t k = k0 + i * blockDim.x;
			if (k < n) row[k] = scale * acc[i];
		}
		return;
	}
	double *red = reinterpret_cast<double *>(buf); // [group][k]
	if (group < groups) red[threadIdx.x] = acc[0];
	__syncthreads();
	for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
		double sum = 0.0;
		for (uint32_t g = 0; g < groups; ++g) sum += red[g * n + k];
		row[k] = scale * sum;
	}
}

// Chains of P = 2 ... 16 sites: a thread per chain, the modes of a wavefront's
// chains added by lane exchanges, one partial row per workgroup of one wavefront.
template <bool DNLS_MODE, int P>
__global__ void __launch_bounds__(64)
k_energy_tiny(const double2 *__restrict__ state, uint32_t copies, const double *__restrict__ omega,
              double *__restrict__ partial) {
	double acc[P];
#pragma unroll
	for (int k = 0; k < P; ++k) acc[k] = 0.0;
	for (uint32_t c = blockIdx.x * 64 + threadIdx.x; c < copies; c += gridDim.x * 64) {
		double2 v[P];
#pragma unroll
		for (int j = 0; j < P; ++j) v[j] = state[size_t(c) * P + j];
		dft_nat<P, -1>(v);
#pragma unroll
		for (int k = 0; k < P; ++k) {
			if constexpr (DNLS_MODE) acc[k] += fma(v[k].x, v[k].x, v[k].y * v[k].y);
			else acc[k] += mode_energy4(v[k], v[(P - k) % P], omega[k]);
		}
	}
#pragma unroll
	for (int k = 0; k < P; ++k) {
		double s = acc[k];
#pragma unroll
		for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w, 64);
		if (threadIdx.x == 0) partial[size_t(blockIdx.x) * P + k] = DNLS_MODE ? s : 0.25 * s;
	}
}

// Workgroup of a chain length: threads, and chains per round.
uint32_t energy_block(const SmoothPlan &pl, uint32_t copies, uint32_t &chains) {
	uint32_t b = choose_block(pl, copies, chains);
	while (b * kModes < pl.n) b *= 2;
	return std::min(b, kMaxBlock);
}

uint32_t energy_groups_per_cu(const SmoothPlan &pl, uint32_t block, uint32_t chains) {
	return std::max(1u, std::min(kLdsBytes / uint32_t(sizeof(double2) * pl.lds_chain * chains), 12 * 64 / block));
}

} // namespace

bool energy_smooth_path(uint32_t n) { return smooth_length(n) || n == 2 || n == 4; }

size_t energy_smooth_table_size(uint32_t n) {
	if (n <= 16) return 0;
	const SmoothPlan pl = make_plan(n);
	return kPlanValues + smooth_twiddles(pl) + (n + 3) / 4;
}

void energy_smooth_table(uint32_t n, double2 *out) {
	if (n <= 16) return;
	const SmoothPlan pl = make_plan(n);
	std::memcpy((void *) out, &pl, sizeof pl);
	smooth_fill_twiddles(pl, out + kPlanValues);
	std::vector<uint32_t> at(n), places(size_t((n + 3) / 4) * 4, 0);
	for (uint32_t e = 0; e < n; ++e) at[smooth_freq(pl, e)] = e + pl.pad * (e / pl.last.d);
	for (uint32_t k = 0; k < n; ++k) places[k] = at[k] | at[k ? n - k : 0] << 16;
	std::memcpy((void *) (out + kPlanValues + smooth_twiddles(pl)), places.data(), sizeof(uint32_t) * places.size());
}

uint32_t energy_smooth_rows(uint32_t n, uint32_t copies) {
	if (n <= 16) return std::min((copies + 63) / 64, 1024u);
	const SmoothPlan pl = make_plan(n);
	uint32_t chains = 1;
	const uint32_t block = energy_block(pl, copies, chains);
	return std::min((copies + chains - 1) / chains, 256 * energy_groups_per_cu(pl, block, chains));
}

hipError_t launch_energy_smooth(hipStream_t st, bool dnls, const double2 *state, uint32_t n, uint32_t copies,
                                const double2 *table, const double *omega, double *partial, uint32_t rows) {
	if (n <= 16) {
#define NLC_F(P)                                                                                                   \
	if (dnls) hipLaunchKernelGGL((k_energy_tiny<true, P>), dim3(rows), dim3(64), 0, st, state, copies, omega, partial); \
	else hipLaunchKernelGGL((k_energy_tiny<false, P>), dim3(rows), dim3(64), 0, st, state, copies, omega, partial)
		NLC_RADIX_SWITCH(16, n, NLC_F)
#undef NLC_F
		return hipGetLastError();
	}
	const SmoothPlan pl = make_plan(n);
	uint32_t chains = 1;
	const uint32_t block = energy_block(pl, copies, chains), ntw = uint32_t(smooth_twiddles(pl));
	// the chains, and the groups' sums at the end
	const size_t lds = std::max(sizeof(double2) * pl.lds_chain * chains, sizeof(double) * block);
	const auto launch = [&](auto *kernel) {
		if (lds > 64 * 1024) {
			const hipError_t e =
			    hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
			if (e != hipSuccess) return e;
		}
		hipLaunchKernelGGL(kernel, dim3(rows), dim3(block), lds, st, state, copies, chains, ntw, table, omega, partial);
		return hipGetLastError();
	};
	return dnls ? launch(k_energy_smooth<true>) : launch(k_energy_smooth<false>);
}

} // namespace nlc
