// Linear-mode energy pass on the register FFT (nlc_fft_reg.inl): chains of 512
// to 4096 sites (powers of two), and through Bluestein's convolution every
// length from 23 to 4096 that has a prime factor above 7.  Reference behaviour
// and formulas as nlc_energy.hip.
//
// Design: N/V threads per chain transform it in registers; mode k needs Z_k and
// Z_{n-k}, which meet in one more LDS exchange; each thread accumulates its V
// modes in registers over the chains of its slot, and the slots of a workgroup
// are added in LDS at the end, one partial row per workgroup.
//
// The powers of two read the state once, 16 B a site, and are bound by that and
// by FP64 issue: the whole pass on 1024 x 16384 takes 108 us (268 MB; 248 with
// the radix-4 Stockham passes through LDS), 512 x 32768 74 (338), 4096 x 4096 142
// (247).  The other lengths took the direct sum over n sites per mode, O(n^2):
// 1001 x 4096 4206 -> 92 us, 101 x 16384 324 -> 49, 4001 x 1024 37.7 ms -> 151 us.
#include "nlc_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

namespace nlc {
namespace {

#include "nlc_dnls_common.inl"
#include "nlc_fft4096.inl"
#include "nlc_fft_reg.inl"

// Values per thread: few, so that the loads of many wavefronts are in flight.
constexpr int energy_values(int N) { return N == 8192 ? 32 : N <= 64 || N == 512 ? 8 : 16; }
template <int N>
using EFft = RegFft<N, energy_values(N)>;

constexpr int kEBlock = 256;

// Partner sums of one part (real or imaginary): acc[s] += (a x_k -+ b x_{n-k})^2.
template <int PART>
__device__ __forceinline__ void add_square(double &acc, double a, double x, double b, double xm) {
	const double e = PART == 0 ? fma(a, x, -b * xm) : fma(a, x, b * xm);
	acc = fma(e, e, acc);
}

// BLUE: n < N/2 + 1 sites through Bluestein's convolution of length N (table:
// bhat in the spectrum's order, the twiddles, the chirp); else N = n (table: the
// twiddles).
// With 16 values per thread three waves per SIMD, two where the real models' both
// transforms spilled for it (42 registers at N = 1024; whole pass 1001 x 4096 96 -> 89 us,
// 2047 x 1024 78 -> 71; without Bluestein two are slower, 1024 x 16384 169 and 201).
template <bool DNLS_MODE, int N, bool BLUE>
__global__ void __launch_bounds__(kEBlock,
                                  (energy_values(N) == 32 ? 2 : energy_values(N) == 16 ? (BLUE && !DNLS_MODE ? 2 : 3) : 4))
k_energy_reg(const double2 *__restrict__ state, uint32_t n_rt, uint32_t copies, const double2 *__restrict__ table,
             const double *__restrict__ omega, double *__restrict__ partial) {
	using F = EFft<N>;
	constexpr int V = F::V;
	constexpr uint32_t T = F::T, kSlots = kEBlock / T;
	static_assert(T <= uint32_t(kEBlock), "");
	extern __shared__ double lds[]; // F::kLds doubles per slot
	const uint32_t n = BLUE ? n_rt : uint32_t(N);
	const uint32_t slot = threadIdx.x / T, t = threadIdx.x % T;
	double *L = lds + F::kLds * slot;
	// the mode of register s, and whether it is one: k = reg_freq(s, t), or with
	// BLUE, where the second transform returns natural order, t + T s
	const auto mode = [&](int s) { return BLUE ? t + T * s : reg_freq<N, V>(s, t); };
	constexpr int VM = BLUE ? V / 2 : V; // modes per thread (n <= N/2)
	double acc[VM];
#pragma unroll
	for (int s = 0; s < VM; ++s) acc[s] = 0.0;
	const uint32_t per_round = kSlots * gridDim.x, rounds = (copies + per_round - 1) / per_round;
	for (uint32_t round = 0; round < rounds; ++round) { // the same for every thread
		const uint32_t c = round * per_round + blockIdx.x * kSlots + slot;
		// the tables are re-read for every chain rather than held in registers
		const double2 *tab = table;
		const double *om = omega;
		asm volatile("" : "+s"(tab), "+s"(om));
		const double2 *tw = BLUE ? tab + N : tab, *chirp = tab + N + F::kTw;
		const bool live = c < copies;
		const double2 *x = state + size_t(live ? c : 0) * n;
		double2 v[V];
#pragma unroll
		for (int j = 0; j < VM; ++j) {
			const uint32_t at = t + T * j;
			v[j] = live && (!BLUE || at < n) ? x[at] : make_double2(0.0, 0.0);
			if (BLUE) v[j] = cmul(v[j], at < n ? chirp[at] : make_double2(0.0, 0.0));
		}
		reg_fft_fwd<N, V, BLUE>(v, L, tw, t);
		if constexpr (BLUE) {
#pragma unroll
			for (int s = 0; s < V; ++s) v[s] = cmul(v[s], tab[T * s + t]);
			reg_fft_inv<N, V>(v, L, tw, t);
			// X_k = w_k C_k; the chirp has modulus 1
			if constexpr (!DNLS_MODE) {
#pragma unroll
				for (int s = 0; s < VM; ++s)
					if (mode(s) < n) v[s] = cmul(v[s], chirp[mode(s)]);
			}
		}
		if constexpr (DNLS_MODE) {
#pragma unroll
			for (int s = 0; s < VM; ++s) acc[s] += fma(v[s].x, v[s].x, v[s].y * v[s].y);
		} else {
			// Z_{n-k}: values stored by (register, thread), or by k with BLUE.  The
			// partner of (s, t) is (V - 1 - s, tp) for every thread but the first of
			// the chain, whose modes pair among themselves (reg_freq).
			const uint32_t h = t / F::r, u = t % F::r;
			const uint32_t tp = F::kThree && h ? (F::r - 1 - u) + F::r * (V - h) : u ? F::r - u : 0;
			const auto partner = [&](int s) -> uint32_t {
				if (BLUE) return mode(s) == 0 || mode(s) >= n ? 0 : n - mode(s);
				const int m = s / F::r, q = s % F::r, mr = V / F::r;
				const int own = ((mr - m) % mr) * F::r + (m ? F::r - 1 - q : (F::r - q) % F::r);
				return t ? T * (V - 1 - s) + tp : T * own;
			};
			reg_sync<N, V>();
			split_exchange([] { reg_sync<N, V>(); },
			    [&](auto p) {
#pragma unroll
				    for (int s = 0; s < VM; ++s)
					    if (!BLUE || mode(s) < n) L[BLUE ? mode(s) : T * s + t] = part_of(v[s], p);
			    },
			    [&](auto p) {
#pragma unroll
				    for (int s = 0; s < VM; ++s) {
					    const double w = BLUE && mode(s) >= n ? 0.0 : om[mode(s)];
					    add_square<decltype(p)::value>(acc[s], 1.0 + w, part_of(v[s], p), 1.0 - w, L[partner(s)]);
				    }
			    });
		}
		// the next chain's first exchange writes slots that other wavefronts may
		// still be reading (the last exchange of this one, or the partners)
		reg_sync<N, V>();
	}
	// the slots' sums in a fixed order, modes in natural order
	__syncthreads();
#pragma unroll
	for (int s = 0; s < VM; ++s)
		if (!BLUE || mode(s) < n) lds[slot * n + mode(s)] = DNLS_MODE ? acc[s] : 0.25 * acc[s];
	__syncthreads();
	for (uint32_t k = threadIdx.x; k < n; k += kEBlock) {
		double sum = 0.0;
#pragma unroll
		for (uint32_t q = 0; q < kSlots; ++q) sum += lds[q * n + k];
		partial[size_t(blockIdx.x) * n + k] = sum;
	}
}

template <int N>
constexpr size_t energy_lds() {
	return sizeof(double) * EFft<N>::kLds * (kEBlock / EFft<N>::T);
}

template <bool DNLS_MODE, int N, bool BLUE>
hipError_t launch_one(hipStream_t st, const double2 *state, uint32_t n, uint32_t copies, const double2 *table,
                      const double *omega, double *partial, uint32_t rows) {
	constexpr size_t lds = energy_lds<N>();
	if (lds > 64 * 1024) {
		const hipError_t e = hipFuncSetAttribute((const void *) k_energy_reg<DNLS_MODE, N, BLUE>,
		                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
		if (e != hipSuccess) return e;
	}
	hipLaunchKernelGGL((k_energy_reg<DNLS_MODE, N, BLUE>), dim3(rows), dim3(kEBlock), lds, st, state, n, copies, table,
	                   omega, partial);
	return hipGetLastError();
}

// Resident workgroups: what the LDS and 2 to 4 wavefronts per SIMD allow on 256 CUs.
template <int N>
uint32_t rows_of(uint32_t copies) {
	constexpr uint32_t kSlots = kEBlock / EFft<N>::T, V = EFft<N>::V;
	constexpr uint32_t by_waves = V == 32 ? 2 : V == 16 ? 3 : 4, by_lds = uint32_t(160 * 1024 / energy_lds<N>());
	return std::min<uint32_t>((copies + kSlots - 1) / kSlots, 256 * std::min(by_waves, by_lds));
}

bool energy_pow2(uint32_t n) { return n >= 512 && n <= 4096 && (n & (n - 1)) == 0; }

// Length of Bluestein's convolution, 0 where it is not used (11 to 22 sites
// keep the direct sum, which is the more accurate there).
uint32_t energy_blue(uint32_t n) {
	if (n < 23 || n > 4096 || (n & (n - 1)) == 0 || smooth_length(n)) return 0;
	uint32_t M = 32;
	while (M < 2 * n - 1) M <<= 1;
	return M;
}

#define NLC_ENERGY_DISPATCH(f, ...)                                                                                \
	if (energy_pow2(n)) switch (n) {                                                                               \
		case 512: return f(512, false)(__VA_ARGS__);                                                                  \
		case 1024: return f(1024, false)(__VA_ARGS__);                                                                \
		case 2048: return f(2048, false)(__VA_ARGS__);                                                                \
		case 4096: return f(4096, false)(__VA_ARGS__);                                                                \
		}                                                                                                             \
	switch (energy_blue(n)) {                                                                                      \
	case 32: return f(32, true)(__VA_ARGS__);                                                                       \
	case 64: return f(64, true)(__VA_ARGS__);                                                                       \
	case 128: return f(128, true)(__VA_ARGS__);                                                                     \
	case 256: return f(256, true)(__VA_ARGS__);                                                                     \
	case 512: return f(512, true)(__VA_ARGS__);                                                                     \
	case 1024: return f(1024, true)(__VA_ARGS__);                                                                   \
	case 2048: return f(2048, true)(__VA_ARGS__);                                                                   \
	case 4096: return f(4096, true)(__VA_ARGS__);                                                                   \
	case 8192: return f(8192, true)(__VA_ARGS__);                                                                   \
	}

template <int N, bool BLUE>
size_t table_values(uint32_t n) {
	return EFft<N>::kTw + (BLUE ? N + n : 0);
}

template <int N, bool BLUE>
void fill_table(uint32_t n, const double2 *blue, double2 *out) {
	using F = EFft<N>;
	if constexpr (BLUE) { // blue: bhat, roots, chirp
		for (uint32_t e = 0; e < uint32_t(N); ++e) out[e] = blue[reg_freq<N, F::V>(e / F::T, e % F::T)];
		std::copy(blue + 2 * size_t(N), blue + 2 * size_t(N) + n, out + N + F::kTw);
		out += N;
	}
	reg_twiddles<N, F::V>(out);
}

} // namespace

bool energy_reg_path(uint32_t n) { return energy_pow2(n) || energy_blue(n); }

size_t energy_reg_table_size(uint32_t n) {
#define NLC_F(N, B) table_values<N, B>
	NLC_ENERGY_DISPATCH(NLC_F, n)
#undef NLC_F
	return 0;
}

uint32_t energy_bluestein_size(uint32_t n) { return energy_blue(n); }

void energy_reg_table(uint32_t n, const double2 *blue, double2 *out) {
#define NLC_F(N, B) fill_table<N, B>
	NLC_ENERGY_DISPATCH(NLC_F, n, blue, out)
#undef NLC_F
}

uint32_t energy_reg_rows(uint32_t n, uint32_t copies) {
#define NLC_F(N, B) rows_of<N>
	NLC_ENERGY_DISPATCH(NLC_F, copies)
#undef NLC_F
	return 0;
}

hipError_t launch_energy_reg(hipStream_t st, bool dnls, const double2 *state, uint32_t n, uint32_t copies,
                             const double2 *table, const double *omega, double *partial, uint32_t rows) {
	if (dnls) {
#define NLC_F(N, B) launch_one<true, N, B>
		NLC_ENERGY_DISPATCH(NLC_F, st, state, n, copies, table, omega, partial, rows)
#undef NLC_F
	} else {
#define NLC_F(N, B) launch_one<false, N, B>
		NLC_ENERGY_DISPATCH(NLC_F, st, state, n, copies, table, omega, partial, rows)
#undef NLC_F
	}
	return hipErrorInvalidValue;
}

} // namespace nlc
