// Plans and sweeps of the in-place FFT of n <= 8192 points with prime factors 2,
// 3, 5 and 7, chains in LDS: shared by the DNLS step and the energy pass.
// n = P_0 P_1 ... P_{m-1} with radices up to 16, as few as there are (1000 = 10 x 10
// x 10).  Pass i of the forward transform takes P_i elements s_i = P_{i+1} ...
// P_{m-1} apart inside blocks of n_i = P_i s_i, transforms them in registers and
// puts them back in place, multiplied by W_{n_i}^{k rest}; the inverse runs the
// same butterflies backwards.  Element k_0 s_0 + k_1 s_1 + ... of the spectrum is
// frequency k_0 + P_0 k_1 + P_0 P_1 k_2 ...  Included inside namespace nlc {
// namespace { ... } } after nlc_fft_smooth.inl.
constexpr int kMaxPasses = 6;
constexpr uint32_t kMaxBlock = 512;

// Division of values below 2^16 by d < 2^14.
struct Magic {
	uint32_t d, m;
	__host__ __device__ Magic() : d(1), m(0) {}
	explicit Magic(uint32_t d_) : d(d_), m(d_ > 1 ? uint32_t((uint64_t(1) << 32) / d_) + 1 : 0) {}
	__host__ __device__ __forceinline__ uint32_t div(uint32_t x) const {
		return d > 1 ? uint32_t((uint64_t(x) * m) >> 32) : x;
	}
};

// LDS address of element e of a chain: e + pad (e / P), P the last radix, with
// pad = 1 for even P, so that the lanes of the inner sweep (P apart) fall in
// different banks.
struct SmoothPass {
	uint32_t radix;
	uint32_t nb;     // butterflies per chain, n / radix
	uint32_t stride; // padded distance of a butterfly's elements
	uint32_t block;  // padded length of a block of n_i elements
	uint32_t tw;     // offset of its twiddles, [k][rest]
	Magic per_chain, per_block; // by nb and by s_i
};
// In device memory behind the tables: read with scalar loads (a kernel argument
// indexed at run time would be copied to scratch).
struct SmoothPlan {
	uint32_t n, m, lds_chain, pad;
	Magic last; // by the last radix
	SmoothPass p[kMaxPasses];
};
constexpr size_t kPlanValues = (sizeof(SmoothPlan) + sizeof(double2) - 1) / sizeof(double2);

// What the sweeps share.
struct SmoothCtx {
	double2 *buf;
	uint32_t chains, lds_chain, pad;
	Magic last;
	const double2 *tw;
};

// The butterflies of one sweep: body(a, address, stride, chain slot's butterfly j,
// rest) for every butterfly of every chain of the workgroup.
template <int P, bool INNER, class Body>
__device__ __forceinline__ void for_butterflies(const SmoothCtx &cx, const SmoothPass &ps, Body body) {
	const uint32_t total = cx.chains * ps.nb;
	uint32_t tid = threadIdx.x;
	asm volatile("" : "+v"(tid)); // the addresses of every sweep are not to be kept in registers over the steps
	for (uint32_t i = tid; i < total; i += blockDim.x) {
		const uint32_t c = ps.per_chain.div(i), j = i - c * ps.nb;
		uint32_t at, rest = 0;
		if (INNER) {
			at = j * (P + cx.pad);
		} else {
			const uint32_t b = ps.per_block.div(j);
			rest = j - b * ps.per_block.d;
			at = b * ps.block + rest + cx.pad * cx.last.div(rest);
		}
		double2 *x = cx.buf + c * cx.lds_chain + at;
		double2 a[P];
#pragma unroll
		for (int k = 0; k < P; ++k) a[k] = x[k * ps.stride];
		body(a, j, rest);
#pragma unroll
		for (int k = 0; k < P; ++k) x[k * ps.stride] = a[k];
	}
}

// Up to this radix a butterfly's factors are read before its DFT, and their
// latency passes behind it; the larger ones have no registers to hold them (20
// steps: 1000 x 2048 2.05 -> 1.98 ms; 1200 x 2048, radix 12 too: the same).
constexpr int kReadAhead = 10;

// a <- f(a), then times the factors w[k s], k = K0 ... P - 1
template <int P, int K0, class F>
__device__ __forceinline__ void then_multiply(double2 *a, const double2 *__restrict__ w, uint32_t s, F f) {
	if constexpr (P <= kReadAhead) {
		double2 t[P];
#pragma unroll
		for (int k = K0; k < P; ++k) t[k] = w[k * s];
		__builtin_amdgcn_sched_barrier(0);
		f(a);
#pragma unroll
		for (int k = K0; k < P; ++k) a[k] = cmul(a[k], t[k]);
	} else {
		f(a);
#pragma unroll
		for (int k = K0; k < P; ++k) {
			a[k] = cmul(a[k], w[k * s]);
			if (k % 8 == 7) __builtin_amdgcn_sched_barrier(0);
		}
	}
}

template <int P>
__device__ __forceinline__ void twiddle_conj(double2 *a, const double2 *__restrict__ tw, uint32_t s) {
#pragma unroll
	for (int k = 1; k < P; ++k) {
		a[k] = cmul(a[k], cconj(tw[k * s]));
		if (k % 8 == 7) __builtin_amdgcn_sched_barrier(0);
	}
}

template <int P, bool INVERSE>
__device__ __forceinline__ void middle(const SmoothCtx &cx, const SmoothPass &ps) {
	for_butterflies<P, false>(cx, ps, [&](double2 *a, uint32_t, uint32_t rest) {
		const double2 *w = cx.tw + ps.tw + rest;
		if constexpr (INVERSE) {
			twiddle_conj<P>(a, w, ps.per_block.d);
			dft_nat<P, +1>(a);
		} else then_multiply<P, 1>(a, w, ps.per_block.d, [](double2 *v) { dft_nat<P, -1>(v); });
	});
}

// f(radix) for the radices up to MAXP, 10 or 16: the registers of a radix 16
// butterfly cost a kernel occupancy or spills also where a plan has none.
#define NLC_RADIX_SWITCH(MAXP, radix, f)                                                                           \
	switch (radix) {                                                                                               \
	case 2: f(2); break;                                                                                           \
	case 3: f(3); break;                                                                                           \
	case 4: f(4); break;                                                                                           \
	case 5: f(5); break;                                                                                           \
	case 6: f(6); break;                                                                                           \
	case 7: f(7); break;                                                                                           \
	case 8: f(8); break;                                                                                           \
	case 9: f(9); break;                                                                                           \
	case 10: f(10); break;                                                                                         \
	default:                                                                                                       \
		if constexpr (MAXP > 10) {                                                                                 \
			if (radix == 12) { f(12); }                                                                            \
			else if (radix == 14) { f(14); }                                                                       \
			else if (radix == 15) { f(15); }                                                                       \
			else { f(16); }                                                                                        \
		}                                                                                                          \
	}

constexpr uint32_t kRadices[] = {16, 15, 14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
// Instructions per point of a pass: the FP64 ones of the DFT and 4 of the
// twiddle, and about 14 per butterfly for its addresses.
double radix_cost(uint32_t p) {
	double dft = 9;
	switch (p) {
	case 2: dft = 2; break;
	case 3: case 4: dft = 4; break;
	case 5: dft = 7.2; break;
	case 6: dft = 6; break;
	case 7: dft = 9.4; break;
	case 8: dft = 6.5; break;
	case 9: dft = 9.8; break;
	case 10: dft = 9.2; break;
	case 12: dft = 8; break;
	case 14: dft = 11.4; break;
	case 15: dft = 11.2; break;
	}
	return dft + 4 + 14.0 / p;
}

// The factorisation of n into `left` radices, descending from max, with the
// fewest operations.
void factor(uint32_t n, uint32_t max, int left, double cost, std::vector<uint32_t> &cur, std::vector<uint32_t> &best,
            double &best_cost) {
	if (!left) {
		if (n == 1 && (best.empty() || cost < best_cost)) best = cur, best_cost = cost;
		return;
	}
	for (const uint32_t p : kRadices) {
		if (p > max || n % p) continue;
		uint64_t reach = 1;
		for (int i = 0; i < left; ++i) reach *= p;
		if (reach < n) return; // and so for every smaller radix
		cur.push_back(p);
		factor(n / p, p, left - 1, cost + radix_cost(p), cur, best, best_cost);
		cur.pop_back();
	}
}

// Radices of n > 16, as few as there are, descending but for an odd one last if
// there is any (its inner sweep needs no padding).
std::vector<uint32_t> radices_of(uint32_t n) {
	std::vector<uint32_t> cur, r;
	double cost = 0;
	for (int m = 2; m <= kMaxPasses && r.empty(); ++m) factor(n, 16, m, 0.0, cur, r, cost);
	for (size_t i = r.size(); i-- > 0;)
		if (r[i] % 2) {
			const uint32_t p = r[i];
			r.erase(r.begin() + i);
			r.push_back(p);
			break;
		}
	return r;
}

SmoothPlan make_plan(uint32_t n) {
	SmoothPlan pl{};
	const std::vector<uint32_t> r = radices_of(n);
	pl.n = n;
	pl.m = uint32_t(r.size());
	const uint32_t last = r.back();
	pl.pad = last % 2 ? 0 : 1;
	pl.last = Magic(last);
	pl.lds_chain = n + pl.pad * (n / last);
	uint32_t ni = n, off = 0;
	for (uint32_t i = 0; i < pl.m; ++i) {
		SmoothPass &p = pl.p[i];
		const uint32_t s = ni / r[i];
		p.radix = r[i];
		p.nb = n / r[i];
		p.stride = i + 1 < pl.m ? s + pl.pad * (s / last) : 1;
		p.block = ni + pl.pad * (ni / last);
		p.tw = off;
		p.per_chain = Magic(p.nb);
		p.per_block = Magic(s);
		if (i + 1 < pl.m) off += ni;
		ni = s;
	}
	return pl;
}

constexpr uint32_t kLdsBytes = 160 * 1024;

// Workgroup of a plan: threads (returned) and chains.  Lanes are idle in the
// last round over the butterflies of a sweep, a CU wants about 9 wavefronts, and
// the wavefronts of a workgroup wait for each other at every sweep; 1, 2, 4 or
// 8 of them, which spread evenly over the SIMDs.  1000 sites, 2048 chains x 20
// steps: 64 threads x 1 chain 1.88 ms, 128 x 2 1.97, 256 x 2 1.86, 512 x 5 (no idle
// lanes, but a single workgroup per CU) 2.37, 320 x 3 2.25, 192 x 1 2.37.  Up to 512
// chains (two per CU) each has its own workgroup, wide enough for one round.
uint32_t choose_block(const SmoothPlan &pl, uint32_t copies, uint32_t &chains) {
	uint32_t most = 0;
	for (uint32_t i = 0; i < pl.m; ++i) most = std::max(most, pl.p[i].nb);
	const uint32_t chain_bytes = pl.lds_chain * uint32_t(sizeof(double2));
	if (copies <= 512) {
		chains = 1;
		return std::min(kMaxBlock, (most + 63) / 64 * 64);
	}
	double best = -1;
	uint32_t best_b = 64;
	for (uint32_t b = 64, step = 0; b <= kMaxBlock; b *= 2, ++step)
		for (uint32_t c = 1; c == 1 || (c * chain_bytes <= kLdsBytes && c * most <= 2 * b); ++c) {
			double used = 0, slots = 0;
			for (uint32_t i = 0; i < pl.m; ++i) {
				const double w = radix_cost(pl.p[i].radix) * pl.p[i].radix;
				used += w * c * pl.p[i].nb;
				slots += w * ((c * pl.p[i].nb + b - 1) / b) * b;
			}
			const uint32_t groups = std::max(1u, std::min(kLdsBytes / (c * chain_bytes), 12 * 64 / b));
			const double waits = (1 - 0.09 * step) * (groups > 1 ? 1.0 : 0.8);
			const double score = used / slots * waits * std::min(1.0, groups * b / (9.0 * 64));
			if (score > best * 1.001) best = score, best_b = b, chains = c;
		}
	return best_b;
}

size_t smooth_twiddles(const SmoothPlan &pl) {
	const SmoothPass &p = pl.p[pl.m - 2];
	return p.tw + size_t(p.per_block.d) * p.radix;
}

void smooth_fill_twiddles(const SmoothPlan &pl, double2 *out) {
	const uint32_t n = pl.n;
	std::vector<double2> w(n); // e^{-2 pi i e/n}
	for (uint32_t e = 0; e <= n / 2; ++e) {
		const double ang = 2.0 * M_PI * double(e) / double(n);
		w[e] = unit_near(std::cos(ang), -std::sin(ang));
		if (e) w[n - e] = make_double2(w[e].x, -w[e].y);
	}
	for (uint32_t i = 0; i + 1 < pl.m; ++i) {
		const uint32_t s = pl.p[i].per_block.d, ni = s * pl.p[i].radix;
		for (uint32_t k = 0; k < pl.p[i].radix; ++k)
			for (uint32_t rest = 0; rest < s; ++rest)
				out[pl.p[i].tw + size_t(k) * s + rest] = w[size_t(k) * rest % ni * (n / ni)];
	}
}

// Frequency of element e of the spectrum.
uint32_t smooth_freq(const SmoothPlan &pl, uint32_t e) {
	uint32_t f = 0, w = 1;
	for (uint32_t i = 0; i < pl.m; ++i) {
		const uint32_t s = pl.p[i].per_block.d;
		f += w * (e / s);
		e %= s;
		w *= pl.p[i].radix;
	}
	return f;
}
