// DNLS split step for chain lengths up to 8192 without a register kernel
// (nlc_dnls.hip, nlc_dnls_reg.hip), chain resident in LDS for a whole batch.
//
// Reference behaviour followed: DNLS.cpp:159-175 (as nlc_dnls.hip).
//
//  * k_dnls_lds: n = 2, 4, 8 and 16, chain in LDS, radix-4 Stockham passes (the
//    inverse transform as conj(FFT(conj(.)))); longer powers of two run in
//    registers (nlc_dnls_reg.hip).
//  * k_dnls_mixed: the other n <= 8192 whose prime factors are 2, 3, 5 and 7
//    (3000, 5000, 6000, ...), the same with the mixed-radix Stockham passes of
//    nlc_fft_mixed.hpp.
#include "nlc_internal.hpp"
#include "nlc_fft_large.hpp"
#include "nlc_fft_mixed.hpp"

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"

// One batch of steps on a chain held in LDS by threads tid < nthr; fft(buf) is
// the forward n-point FFT in place, natural order in and out.  Between substeps
// the buffer holds conj(psi): the inverse transform is conj(FFT(conj(X T))).
// A slot past the last chain (live = false) runs on zeros and writes nothing,
// so that every thread reaches every barrier.
// NT: the thread count as a compile-time constant (0: nthr at run time).
template <uint32_t NT, class Fft>
__device__ __forceinline__ void dnls_lds_batch(double2 *buf, double2 *psi, bool live, uint32_t n, uint32_t tid,
                                               uint32_t nthr_rt, uint32_t steps, const DnlsArgs &a,
                                               const double2 *__restrict__ table, Fft fft) {
	const uint32_t nthr = NT ? NT : nthr_rt;
	for (uint32_t x = tid; x < n; x += nthr) buf[x] = live ? psi[x] : make_double2(0.0, 0.0);
	bool conj_state = false;
	__syncthreads();
	for (uint32_t s = 0; s < steps; ++s) {
		for (int k = 0; k < 7; ++k) {
			const double th = (k == 0 && s) ? a.theta[8] : a.theta[k];
			for (uint32_t x = tid; x < n; x += nthr) {
				const double2 p = conj_state ? cconj(buf[x]) : buf[x];
				buf[x] = nonlinear(p, th);
			}
			__syncthreads();
			fft(buf);
			const double2 *tk = table + size_t(k) * n;
			for (uint32_t j = tid; j < n; j += nthr) buf[j] = cconj(cmul(buf[j], tk[j]));
			__syncthreads();
			fft(buf);
			conj_state = true;
		}
	}
	if (live)
		for (uint32_t x = tid; x < n; x += nthr) {
			const double2 p = conj_state ? cconj(buf[x]) : buf[x];
			psi[x] = nonlinear(p, a.theta[7]);
		}
}

// Threads per chain of k_dnls_lds: n/4 (one radix-4 butterfly per thread and
// pass), kT/(n/4) chains per workgroup.
__host__ __device__ inline uint32_t lds_chain_threads(uint32_t n) { return n >= 4 ? n / 4 : 1u; }

__global__ void __launch_bounds__(kT)
k_dnls_lds(double2 *__restrict__ state, uint32_t n, uint32_t copies, uint32_t steps, DnlsArgs a,
           const double2 *__restrict__ tw, const double2 *__restrict__ table) {
	extern __shared__ double2 buf[];
	const uint32_t nthr = lds_chain_threads(n), per_group = kT / nthr;
	const uint32_t sub = threadIdx.x / nthr, tid = threadIdx.x % nthr;
	const uint32_t chain = blockIdx.x * per_group + sub;
	const bool live = chain < copies;
	dnls_lds_batch<0>(buf + size_t(sub) * n, state + size_t(live ? chain : 0) * n, live, n, tid, nthr, steps, a, table,
	                  [&](double2 *b) { lds_fft_fwd<4 * kT>(b, n, tw, 1, tid, nthr); });
}

// Chains per workgroup of k_dnls_mixed below 512 sites: ceil(n/4) threads per
// chain (no pass then has more than 2 butterflies per thread), kT / that many
// chains; the kT mod nthr threads left over run a dummy slot of their own.
__host__ __device__ inline uint32_t mixed_chain_threads(uint32_t n) { return (n + 3) / 4; }

// SHARED: several chains per workgroup (n <= 512), MAXN = 1024 bounds n per chunk.
template <uint32_t MAXN, bool SHARED>
__global__ void __launch_bounds__(kT)
k_dnls_mixed(double2 *__restrict__ state, uint32_t n, uint32_t copies, uint32_t steps, DnlsArgs a, MixedPlan plan,
             const double2 *__restrict__ tw, const double2 *__restrict__ table) {
	extern __shared__ double2 buf[];
	if constexpr (SHARED) {
		const uint32_t nthr = mixed_chain_threads(n), per_group = kT / nthr;
		const uint32_t sub = threadIdx.x / nthr, tid = threadIdx.x % nthr; // sub == per_group: the dummy slot
		const uint32_t chain = blockIdx.x * per_group + sub;
		const bool live = sub < per_group && chain < copies;
		dnls_lds_batch<0>(buf + size_t(sub) * n, state + size_t(live ? chain : 0) * n, live, n, tid, nthr, steps, a,
		                  table, [&](double2 *b) { mixed::lds_fft<MAXN, kT, false>(b, n, tw, plan, tid, nthr); });
	} else {
		dnls_lds_batch<kT>(buf, state + size_t(blockIdx.x) * n, true, n, threadIdx.x, kT, steps, a, table,
		                   [&](double2 *b) { mixed::lds_fft<MAXN, kT>(b, n, tw, plan); });
	}
}

template <typename K>
hipError_t launch_lds_chain_kernel(K kernel, size_t lds) {
	if (lds > 64 * 1024)
		return hipFuncSetAttribute((const void *) kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
	return hipSuccess;
}

bool pow2(uint32_t n) { return n >= 2 && (n & (n - 1)) == 0; }

// In-place radix-2 FFT on the host (forward sign) in extended precision, for
// bhat: an error of a table entry enters every step alike, so the entries are
// to be good to their last bit.  root[j] = e^{-2 pi i j/n}.
struct Ext {
	long double x, y;
};
void host_fft(std::vector<Ext> &v, const std::vector<Ext> &root) {
	const size_t n = v.size();
	for (size_t i = 1, j = 0; i < n; ++i) {
		size_t bit = n >> 1;
		for (; j & bit; bit >>= 1) j ^= bit;
		j ^= bit;
		if (i < j) std::swap(v[i], v[j]);
	}
	for (size_t len = 2; len <= n; len <<= 1)
		for (size_t b = 0; b < n; b += len)
			for (size_t j = 0; j < len / 2; ++j) {
				const Ext w = root[j * (n / len)];
				Ext &u = v[b + j], &t = v[b + j + len / 2];
				const long double tr = t.x * w.x - t.y * w.y, ti = t.x * w.y + t.y * w.x;
				t = {u.x - tr, u.y - ti};
				u = {u.x + tr, u.y + ti};
			}
}

} // namespace

uint32_t dnls_bluestein_size(uint32_t n) {
	if (n < 2 || pow2(n) || mixed_radix_plan(n, nullptr)) return 0;
	uint32_t M = 1;
	while (M < 2 * n - 1) M <<= 1;
	return M <= kDnlsBluesteinMax ? M : 0;
}

// bhat = FFT_M(b)/M of b_j = conj(w_j) (|j| < n, placed cyclically), the M-point
// roots e^{-2 pi i j/M} and the chirp w_j = e^{-i pi j^2/n}: out[0, M), out[M, 2M),
// out[2M, 2M + n).  With R > 1 bhat is stored in the two-level order [r][k]
// (bhat[r + R k] at r M/R + k).
void bluestein_tables(uint32_t n, uint32_t M, uint32_t R, double2 *out) {
	constexpr long double kPi = 3.141592653589793238462643383279502884L;
	std::vector<Ext> b(M, Ext{0, 0}), root(M);
	for (uint32_t j = 0; j <= M / 8; ++j) { // one octant; the others by symmetry
		long double c, s;
		sincosl(2 * kPi * j / M, &s, &c);
		const uint32_t q = M / 4;
		const Ext z[2] = {{c, -s}, {s, -c}};
		for (uint32_t k = 0; k < 2; ++k) {
			const uint32_t at = k ? q - j : j;
			root[at] = z[k];
			root[at + q] = {z[k].y, -z[k].x};
			root[at + 2 * q] = {-z[k].x, -z[k].y};
			root[(at + 3 * q) % M] = {-z[k].y, z[k].x};
		}
	}
	for (uint32_t j = 0; j < n; ++j) {
		// w_j = e^{-i pi j^2/n}, with j^2 reduced mod 2n so the angle stays in [0, 2 pi)
		long double c, s;
		sincosl(kPi * ((uint64_t(j) * j) % (2 * uint64_t(n))) / n, &s, &c);
		b[j] = {c, s}; // conj(w_j)
		if (j) b[M - j] = b[j];
		out[size_t(2) * M + j] = make_double2(double(c), double(-s)); // w_j
	}
	host_fft(b, root);
	const uint32_t rows = M / R;
	for (uint32_t j = 0; j < M; ++j) {
		const uint32_t at = R > 1 ? (j % R) * rows + j / R : j;
		out[at] = make_double2(double(b[j].x / M), double(b[j].y / M));
		out[M + j] = make_double2(double(root[j].x), double(root[j].y));
	}
}

hipError_t launch_dnls_generic(hipStream_t st, double2 *state, uint32_t n, uint32_t copies, uint32_t steps,
                               const double *theta9, const double2 *tw, const double2 *table) {
	DnlsArgs a;
	for (int i = 0; i < 9; ++i) a.theta[i] = theta9[i];
	if (pow2(n) && n <= kDnlsLdsPow2Max) {
		const uint32_t per_group = kT / lds_chain_threads(n);
		hipLaunchKernelGGL(k_dnls_lds, dim3((copies + per_group - 1) / per_group), dim3(kT),
		                   sizeof(double2) * n * per_group, st, state, n, copies, steps, a, tw, table);
	} else if (MixedPlan plan; mixed_radix_plan(n, &plan)) {
		const uint32_t nthr = mixed_chain_threads(n), per_group = kT / nthr;
		if (per_group > 1) {
			const uint32_t slots = (kT + nthr - 1) / nthr; // with the dummy slot of the left-over threads
			hipLaunchKernelGGL((k_dnls_mixed<4 * kT, true>), dim3((copies + per_group - 1) / per_group), dim3(kT),
			                   sizeof(double2) * n * slots, st, state, n, copies, steps, a, plan, tw, table);
		} else if (n <= 4096) {
			hipLaunchKernelGGL((k_dnls_mixed<4096, false>), dim3(copies), dim3(kT), sizeof(double2) * n, st, state, n,
			                   copies, steps, a, plan, tw, table);
		} else {
			const size_t lds = sizeof(double2) * n;
			hipError_t e = launch_lds_chain_kernel(k_dnls_mixed<kDnlsLdsMax, false>, lds);
			if (e != hipSuccess) return e;
			hipLaunchKernelGGL((k_dnls_mixed<kDnlsLdsMax, false>), dim3(copies), dim3(kT), lds, st, state, n, copies, steps,
			                   a, plan, tw, table);
		}
	} else {
		return hipErrorInvalidValue;
	}
	return hipGetLastError();
}

} // namespace nlc
