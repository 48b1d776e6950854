// Linear-mode energy pass of chains up to 65536 sites whose prime factors are 2,
// 3, 5 and 7 (the powers of two from 8 to 4096 have their own kernels).  Reference
// behaviour and formulas as nlc_energy.hip.
//
// Design: several chains per workgroup in LDS, transformed by the in-place
// sweeps of nlc_smooth_plan.inl; mode k of a chain is read from the place of Z_k
// (and of Z_{n-k}, real models) through a table of places, and each thread
// accumulates its modes over the chains in registers.  Up to 16 sites a thread
// transforms a whole chain in registers; from 8192 sites on a workgroup transforms
// two rows of a chain (k_energy_rows).
//
// Bound by the latency of the sweeps, as the DNLS kernel; the state is read once.
// Whole pass at 4.2 million sites (67 MB), against one chain per workgroup with
// radix 2, 3, 4, 5 and 7 Stockham passes: 20 sites 72 us (1154), 48 60 (618), 100 63
// (355), 360 70 (173), 1000 65 (105), 5000 80 (167), 7000 82 (167); 12 x 300000 32
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

// The forward transform of the chains in LDS.
__device__ __forceinline__ void transform(const SmoothCtx &cx, const SmoothPlan *plan, uint32_t m) {
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
		transform(cx, plan, m); // chains past the last one too (whatever they hold), which are not read
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

// Longer chains, n = R C with R <= 16 rows of C <= kRowMax sites.  Mode r + R f is
// mode f of row r, y_r[c] = W_n^{c r} sum_j x[c + C j] W_R^{j r}.  A workgroup takes
// the rows r and R - r (or 0 and R/2; 0 alone for odd R), which hold each other's
// modes -k, so the transform never leaves LDS: the row sums are formed while the
// chain is read, once per pair of rows, most of them from the caches.  Bound by
// the latency of the sweeps between barriers, with the one workgroup per CU that two
// rows' LDS leaves (two of 256 threads where the rows are short: the same time);
// about 2.5 times the time of one read of the state.
// The whole pass, before (two-level FFT or Bluestein's two transforms through HBM)
// and with this: 20000 sites x 256 chains 395 -> 111 us, 10000 x 420 334 -> 101, 12000 x
// 350 288 -> 104, 24000 x 200 360 -> 144, 16384 x 256 160 -> 103, 65536 x 32 156 -> 119,
// 8192 x 512 (one workgroup per chain, in LDS) 127 -> 102.
struct RowsHead {
	uint32_t R, C, units, ntw;
};
constexpr uint32_t kRowMax = 4096; // kModes values per thread, and two rows fit the LDS

// table: the plan of C (kPlanValues), RowsHead, per unit R pairs of coefficients,
// the factors W_n^{c r} as [r][c], the twiddles of C (ntw), the places of the modes
// of a row, 4 to a value.
template <bool DNLS_MODE>
__global__ void __launch_bounds__(kMaxBlock, 2)
k_energy_rows(const double2 *__restrict__ state, uint32_t copies, uint32_t rows, const double2 *__restrict__ table,
              const double *__restrict__ omega, double *__restrict__ partial) {
	extern __shared__ double2 buf[];
	const SmoothPlan *plan = reinterpret_cast<const SmoothPlan *>(table);
	const RowsHead *head = reinterpret_cast<const RowsHead *>(table + kPlanValues);
	const uint32_t R = head->R, C = head->C, U = head->units, n = R * C, m = plan->m;
	// the units of one row of partial on one XCD (workgroups go round the 8 XCDs)
	const uint32_t turn = blockIdx.x / (8 * U), u = blockIdx.x / 8 % U, g = turn * 8 + blockIdx.x % 8;
	if (g >= rows) return;
	const double2 *coef = table + kPlanValues + 1 + u * R, *factors = table + kPlanValues + 1 + U * R;
	const bool self = u == 0;
	const uint32_t pair = self ? R / 2 : R - u, chains = self && R % 2 ? 1 : 2;
	const SmoothCtx cx{buf, chains, plan->lds_chain, plan->pad, plan->last, factors + n};
	const uint32_t *places = reinterpret_cast<const uint32_t *>(factors + n + head->ntw);
	double acc[kModes];
#pragma unroll
	for (int i = 0; i < kModes; ++i) acc[i] = 0.0;
	for (uint32_t copy = g; copy < copies; copy += rows) {
		const double2 *z = state + size_t(copy) * n;
		for (uint32_t c = threadIdx.x; c < C; c += blockDim.x) {
			double2 a = make_double2(0.0, 0.0), b = a;
#pragma unroll 8
			for (uint32_t j = 0; j < R; ++j) {
				const double2 x = z[c + C * j], w = coef[j];
				a = make_double2(fma(w.x, x.x, a.x), fma(w.x, x.y, a.y));
				b = make_double2(fma(w.y, x.x, b.x), fma(w.y, x.y, b.y));
			}
			if (!self) b = make_double2(b.y, -b.x); // cosines and sines: W^{j r} = cos - i sin
			double2 *x = buf + c + cx.pad * cx.last.div(c);
			x[0] = cmul(cadd(a, b), factors[u * C + c]);
			if (chains == 2) x[cx.lds_chain] = cmul(csub(a, b), factors[pair * C + c]);
		}
		__syncthreads();
		transform(cx, plan, m);
#pragma unroll
		for (int i = 0; i < kModes; ++i) {
			const uint32_t s = threadIdx.x + i * blockDim.x;
			if (s >= chains * C) break;
			const uint32_t second = s >= C, f = s - second * C, r = second ? pair : u;
			// -k is in the other row, or in this one (0 to itself)
			const uint32_t back = r == 0 ? (f ? C - f : 0) : C - 1 - f, row = self ? second : 1 - second;
			const double2 v = buf[second * cx.lds_chain + places[f]];
			if constexpr (DNLS_MODE) acc[i] += fma(v.x, v.x, v.y * v.y);
			else acc[i] += mode_energy4(v, buf[row * cx.lds_chain + places[back]], omega[r + R * f]);
		}
		__syncthreads();
	}
	double *out = partial + size_t(g) * n;
#pragma unroll
	for (int i = 0; i < kModes; ++i) {
		const uint32_t s = threadIdx.x + i * blockDim.x;
		if (s >= chains * C) break;
		const uint32_t second = s >= C;
		out[(second ? pair : u) + R * (s - second * C)] = (DNLS_MODE ? 1.0 : 0.25) * acc[i];
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

namespace {

// Rows of a chain above 8192 sites (8192 too) with prime factors 2, 3, 5, 7; 0 if
// there is no such split (n > 65536, or 59049).  The fewest, for each pair of rows
// reads the chain (24000 x 200: 6 rows 144 us, 12 rows 186), and an even number, for
// row 0 alone leaves its workgroup half empty (20000 x 256: 5 rows 143 us, 8 rows 111).
uint32_t energy_row_count(uint32_t n) {
	if (n < 8192 || n > 16 * kRowMax) return 0;
	uint32_t odd = n;
	for (const uint32_t f : {2u, 3u, 5u, 7u})
		while (odd % f == 0) odd /= f;
	if (odd != 1) return 0;
	for (uint32_t first = 4; first >= 3; --first)
		for (uint32_t R = first; R <= 16; R += 2)
			if (n % R == 0 && n / R <= kRowMax && 2 * sizeof(double2) * make_plan(n / R).lds_chain <= kLdsBytes) return R;
	return 0;
}

} // namespace

bool energy_smooth_path(uint32_t n) { return smooth_length(n) || n == 2 || n == 4 || energy_row_count(n); }

size_t energy_smooth_table_size(uint32_t n) {
	if (n <= 16) return 0;
	if (const uint32_t R = energy_row_count(n)) {
		const uint32_t C = n / R;
		return kPlanValues + 1 + size_t((R + 1) / 2) * R + n + smooth_twiddles(make_plan(C)) + (C + 3) / 4;
	}
	const SmoothPlan pl = make_plan(n);
	return kPlanValues + smooth_twiddles(pl) + (n + 3) / 4;
}

void energy_smooth_table(uint32_t n, double2 *out) {
	if (n <= 16) return;
	if (const uint32_t R = energy_row_count(n)) {
		const uint32_t C = n / R, U = (R + 1) / 2;
		const SmoothPlan pl = make_plan(C);
		std::memcpy((void *) out, &pl, sizeof pl);
		const RowsHead head{R, C, U, uint32_t(smooth_twiddles(pl))};
		std::memcpy((void *) (out + kPlanValues), &head, sizeof head);
		out += kPlanValues + 1;
		for (uint32_t u = 0; u < U; ++u)
			for (uint32_t j = 0; j < R; ++j) {
				const double ang = 2.0 * M_PI * double(u * j % R) / double(R);
				// rows 0 and R/2: the sums over even and odd j (0 alone: over all)
				*out++ = u ? make_double2(std::cos(ang), std::sin(ang))
				           : make_double2(R % 2 || j % 2 == 0 ? 1.0 : 0.0, R % 2 || j % 2 == 0 ? 0.0 : 1.0);
			}
		for (uint32_t r = 0; r < R; ++r)
			for (uint32_t c = 0; c < C; ++c) {
				const double ang = 2.0 * M_PI * double(uint64_t(r) * c % n) / double(n);
				*out++ = make_double2(std::cos(ang), -std::sin(ang));
			}
		smooth_fill_twiddles(pl, out);
		std::vector<uint32_t> places(size_t((C + 3) / 4) * 4, 0);
		for (uint32_t e = 0; e < C; ++e) places[smooth_freq(pl, e)] = e + pl.pad * (e / pl.last.d);
		std::memcpy((void *) (out + head.ntw), places.data(), sizeof(uint32_t) * places.size());
		return;
	}
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
	if (const uint32_t R = energy_row_count(n)) {
		// time in passes over a chain: the rounds of 256 workgroups, and a row of partial
		// written and read back; at most 256 MiB of rows
		const uint32_t U = (R + 1) / 2, most = std::min({copies, 1024u, (1u << 25) / n});
		uint32_t best = 1;
		double least = 1e300;
		for (uint32_t g = 1; g <= most; ++g) {
			const double t = 256.0 * ((g * U + 255) / 256) * ((copies + g - 1) / g) + g;
			if (t < least) least = t, best = g;
		}
		return best;
	}
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
	if (const uint32_t R = energy_row_count(n)) {
		const size_t lds = 2 * sizeof(double2) * make_plan(n / R).lds_chain;
		const auto kernel = dnls ? k_energy_rows<true> : k_energy_rows<false>;
		const hipError_t e = hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
		if (e != hipSuccess) return e;
		hipLaunchKernelGGL(kernel, dim3((rows + 7) / 8 * 8 * ((R + 1) / 2)), dim3(kMaxBlock), lds, st, state, copies, rows,
		                   table, omega, partial);
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
