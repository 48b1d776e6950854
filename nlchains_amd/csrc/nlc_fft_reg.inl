// Register FFT of N = 32 ... 16384 points (powers of two), FP64: N/V threads x V
// values per chain, V = 8, 16 or 32.  Passes of V over the strided values of a
// thread, a last one of the r points that are left:
//   two passes   N = V r          64 = 8 x 8, 256 = 16 x 16, 512 = 32 x 16, 1024 = 32 x 32
//   three passes N = V V r        512 = 8 x 8 x 8, 4096 = 16 x 16 x 16, 16384 = 32 x 32 x 16
// so the data passes through LDS once or twice per transform; where a chain's
// threads lie in one wavefront the exchanges need no workgroup barrier.
// Decimation in frequency forward, in time backward: the spectrum stays in a
// permuted order that the caller's tables follow (reg_freq).
//
// The inverse is the conjugate transpose of the forward transform, stage by
// stage, so that over many steps only the moduli of the twiddles matter: a
// twiddle that is off the unit circle scales its points in every step alike.
// The twiddles therefore come from tables, in the order of use, of roots rounded
// to lie on the unit circle; running powers (a few ulp off) made the error after
// 30 steps 2 to 4 times as large.
// Included inside namespace nlc { namespace { ... } } after nlc_fft4096.inl.

// position of element k of an 8-point transform in "transposed" order
__host__ __device__ constexpr int pos8(int k) { return 4 * (k & 1) + (k >> 1); }

// z * exp(SIGN 2 pi i j / 8), j = 0..3
template <int SIGN, int J>
__device__ __forceinline__ double2 w8mul(double2 z) {
	constexpr double h = half_root<SIGN, double>;
	if constexpr (J == 0) return z;
	else if constexpr (J == 2) return SIGN < 0 ? make_double2(z.y, -z.x) : make_double2(-z.y, z.x);
	else if constexpr (J == 1) {
		return SIGN < 0 ? make_double2(h * (z.x + z.y), h * (z.y - z.x)) : make_double2(h * (z.x - z.y), h * (z.x + z.y));
	} else {
		return SIGN < 0 ? make_double2(h * (z.y - z.x), -h * (z.x + z.y)) : make_double2(-h * (z.x + z.y), h * (z.x - z.y));
	}
}

// 8-point DFT, natural in -> transposed out: radix-2 butterflies (j, j + 4)
// with twiddles W8^j, then DFT4 of the sums (even outputs, registers 0..3)
// and of the differences (odd outputs, registers 4..7).
template <int SIGN>
__device__ __forceinline__ void dft8_n2t(double2 v[8]) {
	double2 d[4];
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		d[j] = csub(v[j], v[j + 4]);
		v[j] = cadd(v[j], v[j + 4]);
	}
	v[4] = d[0];
	v[5] = w8mul<SIGN, 1>(d[1]);
	v[6] = w8mul<SIGN, 2>(d[2]);
	v[7] = w8mul<SIGN, 3>(d[3]);
	dft4<SIGN>(v[0], v[1], v[2], v[3]);
	dft4<SIGN>(v[4], v[5], v[6], v[7]);
}

// transposed in -> natural out (decimation in time): DFT4 of the even and of
// the odd elements, twiddle the odd ones by W8^j, butterflies (j, j + 4).
template <int SIGN>
__device__ __forceinline__ void dft8_t2n(double2 v[8]) {
	dft4<SIGN>(v[0], v[1], v[2], v[3]);
	dft4<SIGN>(v[4], v[5], v[6], v[7]);
	const double2 o[4] = {v[4], w8mul<SIGN, 1>(v[5]), w8mul<SIGN, 2>(v[6]), w8mul<SIGN, 3>(v[7])};
#pragma unroll
	for (int j = 0; j < 4; ++j) {
		v[j + 4] = csub(v[j], o[j]);
		v[j] = cadd(v[j], o[j]);
	}
}

// exp(SIGN 2 pi i j/32), j < 16, correctly rounded (but for half_root)
template <int SIGN>
__device__ __forceinline__ constexpr double w32c(int j) {
	constexpr double c[9] = {1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
	                         half_root<SIGN, double>, 0.55557023301960222474, 0.38268343236508977173,
	                         0.19509032201612826785, 0.0};
	return j <= 8 ? c[j] : -c[16 - j];
}
template <int SIGN>
__device__ __forceinline__ constexpr double w32s(int j) {
	return SIGN * w32c<SIGN>(j <= 8 ? 8 - j : j - 8);
}

// 32-point DFT in registers as two 16-point ones.  Permuted order: element k at
// pos32(k).  natural -> permuted: butterflies (j, j + 16), twiddle W32^j on the
// differences (the odd outputs).
__host__ __device__ constexpr int pos32(int k) { return 16 * (k & 1) + pos(k >> 1); }

template <int SIGN>
__device__ __forceinline__ void dft32_n2p(double2 v[32]) {
#pragma unroll
	for (int j = 0; j < 16; ++j) {
		const double2 d = csub(v[j], v[j + 16]);
		v[j] = cadd(v[j], v[j + 16]);
		if (j == 0) v[j + 16] = d;
		else if (j == 8) v[j + 16] = make_double2(-SIGN * d.y, SIGN * d.x);
		else v[j + 16] = cmul(d, make_double2(w32c<SIGN>(j), w32s<SIGN>(j)));
	}
	dft16_n2t<SIGN>(v);
	dft16_n2t<SIGN>(v + 16);
}

// permuted -> natural: E and O of the even and odd elements, then E +- W32^j O.
template <int SIGN>
__device__ __forceinline__ void dft32_p2n(double2 v[32]) {
	dft16_t2n<SIGN>(v);
	dft16_t2n<SIGN>(v + 16);
#pragma unroll
	for (int j = 0; j < 16; ++j) {
		double2 o = v[j + 16];
		if (j == 8) o = make_double2(-SIGN * o.y, SIGN * o.x);
		else if (j) o = cmul(o, make_double2(w32c<SIGN>(j), w32s<SIGN>(j)));
		v[j + 16] = csub(v[j], o);
		v[j] = cadd(v[j], o);
	}
}

// natural -> permuted DFT of V = 8, 16 or 32 values of which the upper half is
// zero (not read): the first butterflies copy.
template <int V, int SIGN>
__device__ __forceinline__ void dft_n2p_half(double2 *v) {
	if constexpr (V == 32) {
#pragma unroll
		for (int j = 0; j < 16; ++j) {
			if (j == 0) v[16] = v[0];
			else if (j == 8) v[j + 16] = make_double2(-SIGN * v[j].y, SIGN * v[j].x);
			else v[j + 16] = cmul(v[j], make_double2(w32c<SIGN>(j), w32s<SIGN>(j)));
		}
		dft16_n2t<SIGN>(v);
		dft16_n2t<SIGN>(v + 16);
	} else if constexpr (V == 16) {
#pragma unroll
		for (int b = 0; b < 4; ++b) { // DFT4 of (a0, a1, 0, 0)
			const double2 a0 = v[b], a1 = v[4 + b], i1 = make_double2(-SIGN * a1.y, SIGN * a1.x);
			v[b] = cadd(a0, a1);
			v[4 + b] = cadd(a0, i1);
			v[8 + b] = csub(a0, a1);
			v[12 + b] = csub(a0, i1);
		}
		dft4<SIGN>(v[0], v[1], v[2], v[3]);
		dft4_tw<SIGN, 1>(v[4], v[5], v[6], v[7]);
		dft4_tw<SIGN, 2>(v[8], v[9], v[10], v[11]);
		dft4_tw<SIGN, 3>(v[12], v[13], v[14], v[15]);
	} else {
		static_assert(V == 8, "");
		v[4] = v[0];
		v[5] = w8mul<SIGN, 1>(v[1]);
		v[6] = w8mul<SIGN, 2>(v[2]);
		v[7] = w8mul<SIGN, 3>(v[3]);
		dft4<SIGN>(v[0], v[1], v[2], v[3]);
		dft4<SIGN>(v[4], v[5], v[6], v[7]);
	}
}

// R-point DFTs, R = 2, 4, 8, 16, 32, with element k of the permuted side at
// perm<R>(k).
template <int R>
__host__ __device__ constexpr int perm(int k) {
	return R == 32 ? pos32(k) : R == 16 ? pos(k) : R == 8 ? pos8(k) : k;
}
template <int R, int SIGN>
__device__ __forceinline__ void dft_n2p(double2 *v) {
	if constexpr (R == 32) dft32_n2p<SIGN>(v);
	else if constexpr (R == 16) dft16_n2t<SIGN>(v);
	else if constexpr (R == 8) dft8_n2t<SIGN>(v);
	else if constexpr (R == 4) dft4<SIGN>(v[0], v[1], v[2], v[3]);
	else {
		const double2 d = csub(v[0], v[1]);
		v[0] = cadd(v[0], v[1]);
		v[1] = d;
	}
}
template <int R, int SIGN>
__device__ __forceinline__ void dft_p2n(double2 *v) {
	if constexpr (R == 32) dft32_p2n<SIGN>(v);
	else if constexpr (R == 16) dft16_t2n<SIGN>(v);
	else if constexpr (R == 8) dft8_t2n<SIGN>(v);
	else dft_n2p<R, SIGN>(v);
}

// Geometry.  T threads per chain; the last exchange runs in groups of r
// threads.  LDS per chain: one row of G doubles per group, G an odd multiple
// of r.  First exchange of three passes: element (t, k0) at G k0 + t.  Last
// exchange: element (u, k) of a group at u + (r + 1) k of its row, or for r <= 4
// at r k + (u xor k mod r), which needs no padding.  The 8-byte accesses of 32
// consecutive lanes then fall in different bank pairs: consecutive t; u + G h,
// where G h runs over the multiples of r; (r + 1) u + G h with r + 1 odd, or
// r u + (q xor u) + G h.
template <int N, int V_>
struct RegFft {
	static_assert(N >= 32 && N <= 16384 && (N & (N - 1)) == 0, "");
	static constexpr int V = V_;
	static constexpr uint32_t T = N / V;
	static constexpr bool kThree = T > uint32_t(V);
	static constexpr int r = kThree ? int(T) / V : int(T);
	static constexpr bool kXor = r <= 4;
	static constexpr uint32_t G = kXor ? r * (V + 1) : r * (((V * (r + 1) + r - 1) / r) | 1);
	static constexpr uint32_t kLds = (kThree ? V : 1) * G; // doubles per chain
	static constexpr uint32_t kBlock = T > 64 ? T : 64, kChains = kBlock / T;
	// from 2048 points on twiddles as products of two table entries (twiddle_table)
	static constexpr int kProd = N < 2048 ? 0 : V == 32 ? 8 : 4;
	// tables: tw1[k0 T + t] = W_N^{t k0}, then (three passes) tw2[k1 r + u] = W_T^{u k1}
	static constexpr uint32_t kTw = N + (kThree ? V * r : 0);
};

// Frequency of the value in register s of thread t after the forward transform.
template <int N, int V>
__host__ __device__ constexpr uint32_t reg_freq(uint32_t s, uint32_t t) {
	using F = RegFft<N, V>;
	const uint32_t k1 = t % F::r + F::r * (s / F::r), k2 = s % F::r;
	return F::kThree ? t / F::r + F::V * k1 + F::V * F::V * k2 : k1 + F::V * k2;
}

// Exchange barrier: a wavefront's LDS operations complete in order, so chains
// inside one need only keep the compiler from reordering them.
template <int N, int V>
__device__ __forceinline__ void reg_sync() {
	if constexpr (RegFft<N, V>::T > 64) lds_barrier();
	else wave_sync();
}

// Real, then imaginary parts through LDS (half the LDS, so twice the chains per
// CU): write and read get the part as an integral constant.  The real pass
// touches only the .x halves, so the .y halves still hold the imaginary parts
// in the old order.
template <class SyncF, class W, class Rd>
__device__ __forceinline__ void split_exchange(SyncF sync, W write, Rd read) {
	write(std::integral_constant<int, 0>());
	sync();
	read(std::integral_constant<int, 0>());
	sync();
	write(std::integral_constant<int, 1>());
	sync();
	read(std::integral_constant<int, 1>());
}
template <class P>
__device__ __forceinline__ double &part_of(double2 &z, P) {
	if constexpr (P::value == 0) return z.x;
	else return z.y;
}

// Slots of the last exchange seen by thread u of a group: mine(k) is element
// (u, k), other(m, q) is element (q, u + r m).
template <int N, int V>
struct RegRow {
	using F = RegFft<N, V>;
	static constexpr int r = F::r;
	double *a[F::kXor ? r : 1], *b[F::kXor ? r : 1];
	__device__ __forceinline__ RegRow(double *row, uint32_t u) {
		if constexpr (F::kXor) {
#pragma unroll
			for (int c = 0; c < r; ++c) a[c] = row + (u ^ c), b[c] = row + r * u + (u ^ c);
		} else {
			a[0] = row + u;
			b[0] = row + (r + 1) * u;
		}
	}
	__device__ __forceinline__ double &mine(int k) const {
		if constexpr (F::kXor) return a[k % r][r * k];
		else return a[0][(r + 1) * k];
	}
	__device__ __forceinline__ double &other(int m, int q) const {
		if constexpr (F::kXor) return b[q][r * r * m];
		else return b[0][q + (r + 1) * r * m];
	}
};

// v[at(k)] *= tw[stride k] (conjugated when CONJ), k = 1 ... V - 1.  PROD > 0:
// entry h + k (h a multiple of PROD, k < PROD) as the product of entries h and k,
// PROD - 1 + V/PROD - 1 loads instead of V - 1: the tables of the longer
// transforms come from L2, and their loads were what the kernels waited for
// (8192 sites x 512, 20 steps: 4.40 -> 3.09 ms; 16384 x 256 4.44 -> 3.57; 4096 x
// 4096 10.08 -> 9.5; 2048 x 2048 2.90 -> 2.78).  The products raise the error
// after 30 steps by a quarter to a half (4096 sites 1.9e-14 -> 2.9e-14), so up to
// 1024 points, where they gain nothing, the entries are read.
template <int V, bool CONJ, bool PERM, int PROD>
__device__ __forceinline__ void twiddle_table(double2 *v, const double2 *__restrict__ tw, uint32_t stride) {
	constexpr int B = PROD ? PROD : V;
	double2 lo[B];
#pragma unroll
	for (int h = 0; h < V; h += B) {
		double2 hi = make_double2(1.0, 0.0);
		if (h) hi = CONJ ? cconj(tw[stride * h]) : tw[stride * h];
#pragma unroll
		for (int k = 0; k < B; ++k) {
			if (h + k == 0) continue;
			if (h == 0) lo[k] = CONJ ? cconj(tw[stride * k]) : tw[stride * k];
			const double2 w = h == 0 ? lo[k] : k == 0 ? hi : cmul(hi, lo[k]);
			const int at = PERM ? perm<V>(h + k) : h + k;
			v[at] = cmul(v[at], w);
		}
	}
}

// Forward: x[t + T j] at v[j] in, X[reg_freq(s, t)] at v[s] out.  t: the thread
// in its chain, L: the chain's kLds doubles.  LDS hazards as for
// fft4096_fwd_split: the first slots a thread writes in an exchange are ones it
// (or its wavefront, in its own rows) read last.
// HALF: x is zero from N/2 on (v[V/2 ...] is not read).
template <int N, int V, bool HALF = false>
__device__ __forceinline__ void reg_fft_fwd(double2 *v, double *L, const double2 *__restrict__ tw, uint32_t t) {
	using F = RegFft<N, V>;
	constexpr int r = F::r;
	const uint32_t u = t % r, h = t / r; // two passes: h = 0
	if constexpr (HALF) dft_n2p_half<V, -1>(v);
	else dft_n2p<V, -1>(v);
	twiddle_table<V, false, true, F::kProd>(v, tw + t, F::T);
	const RegRow<N, V> row(L + F::G * h, u);
	if constexpr (F::kThree) {
		double *w = L + t;
		const double *g = L + F::G * h + u;
		split_exchange([] { reg_sync<N, V>(); },
		    [&](auto p) {
#pragma unroll
			    for (int k0 = 0; k0 < V; ++k0) w[F::G * k0] = part_of(v[perm<V>(k0)], p);
		    },
		    [&](auto p) {
#pragma unroll
			    for (int j = 0; j < V; ++j) part_of(v[perm<V>(j)], p) = g[r * j];
		    });
		dft_p2n<V, -1>(v);
		twiddle_table<V, false, false, F::kProd>(v, tw + N + u, r);
	}
	wave_sync();
	split_exchange([] { wave_sync(); },
	    [&](auto p) {
#pragma unroll
		    for (int k = 0; k < V; ++k) row.mine(k) = part_of(v[F::kThree ? k : perm<V>(k)], p);
	    },
	    [&](auto p) {
#pragma unroll
		    for (int m = 0; m < V / r; ++m)
#pragma unroll
			    for (int q = 0; q < r; ++q) part_of(v[m * r + perm<r>(q)], p) = row.other(m, q);
	    });
#pragma unroll
	for (int m = 0; m < V / r; ++m) dft_p2n<r, -1>(v + m * r);
}

// Inverse (unnormalised), the conjugate transpose of reg_fft_fwd.
template <int N, int V>
__device__ __forceinline__ void reg_fft_inv(double2 *v, double *L, const double2 *__restrict__ tw, uint32_t t) {
	using F = RegFft<N, V>;
	constexpr int r = F::r;
	const uint32_t u = t % r, h = t / r;
#pragma unroll
	for (int m = 0; m < V / r; ++m) dft_n2p<r, +1>(v + m * r);
	const RegRow<N, V> row(L + F::G * h, u);
	wave_sync();
	split_exchange([] { wave_sync(); },
	    [&](auto p) {
#pragma unroll
		    for (int m = 0; m < V / r; ++m)
#pragma unroll
			    for (int q = 0; q < r; ++q) row.other(m, q) = part_of(v[m * r + perm<r>(q)], p);
	    },
	    [&](auto p) {
#pragma unroll
		    for (int k = 0; k < V; ++k) part_of(v[perm<V>(k)], p) = row.mine(k);
	    });
	if constexpr (F::kThree) {
		twiddle_table<V, true, true, F::kProd>(v, tw + N + u, r);
		dft_p2n<V, +1>(v);
		double *w = L + F::G * h + u;
		const double *g = L + t;
		wave_sync();
		split_exchange([] { reg_sync<N, V>(); },
		    [&](auto p) {
#pragma unroll
			    for (int j = 0; j < V; ++j) w[r * j] = part_of(v[j], p);
		    },
		    [&](auto p) {
#pragma unroll
			    for (int k0 = 0; k0 < V; ++k0) part_of(v[perm<V>(k0)], p) = g[F::G * k0];
		    });
	}
	twiddle_table<V, true, true, F::kProd>(v, tw + t, F::T);
	dft_p2n<V, +1>(v);
}

// Of the neighbours of a rounded cosine and sine the pair closest to the unit
// circle (the angle moves by an ulp at most, which a transform and its inverse
// cancel).
inline double2 unit_near(double c, double s) {
	double2 best = make_double2(c, s);
	if (c == 0 || s == 0) return best;
	long double least = std::fabs((long double) c * c + (long double) s * s - 1);
	for (const double ci : {std::nextafter(c, -2.0), c, std::nextafter(c, 2.0)})
		for (const double si : {std::nextafter(s, -2.0), s, std::nextafter(s, 2.0)}) {
			const long double off = std::fabs((long double) ci * ci + (long double) si * si - 1);
			if (off < least) least = off, best = make_double2(ci, si);
		}
	return best;
}

// e^{-2 pi i e/n}, e < n (n a multiple of 8).  One octant; the others by symmetry.
inline std::vector<double2> unit_roots(uint32_t n) {
	std::vector<double2> w(n);
	for (uint32_t e = 0; e <= n / 8; ++e) {
		const double ang = 2.0 * M_PI * double(e) / double(n);
		const double2 u = unit_near(std::cos(ang), -std::sin(ang));
		const uint32_t q = n / 4;
		// quarter turns of u and of its mirror image at q - e
		const double2 z[2] = {u, make_double2(-u.y, -u.x)};
		for (uint32_t k = 0; k < 2; ++k) {
			const uint32_t at = k ? q - e : e;
			w[at] = z[k];
			w[at + q] = make_double2(z[k].y, -z[k].x);
			w[at + 2 * q] = make_double2(-z[k].x, -z[k].y);
			w[(at + 3 * q) % n] = make_double2(-z[k].y, z[k].x);
		}
	}
	return w;
}

// The twiddle tables tw1 and tw2 of RegFft (kTw values).
template <int N, int V>
void reg_twiddles(double2 *out) {
	using F = RegFft<N, V>;
	const std::vector<double2> w = unit_roots(N);
	for (uint32_t e = 0; e < N; ++e) out[e] = w[(e / F::T) * (e % F::T) % N];
	for (uint32_t e = 0; e < F::kTw - N; ++e) out[N + e] = w[(e / F::r) * (e % F::r) * V % N];
}
