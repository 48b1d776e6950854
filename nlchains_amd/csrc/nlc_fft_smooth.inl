// DFTs of P points in registers, P = 2 ... 16 with prime factors 2, 3, 5, 7:
// natural order in and out.  Primes from their symmetric form (sums and
// differences of x_j and x_{P-j}), coprime products by the prime factor map
// (Good 1958; no twiddles), 8 and 16 as in nlc_fft4096.inl / nlc_fft_reg.inl.
// Included inside namespace nlc { namespace { ... } } after nlc_fft_reg.inl.

// cos and sin of 2 pi j/P, P = 3, 5, 7, 9, rounded to nearest
template <int P>
__device__ __forceinline__ constexpr double rootc(int j) {
	constexpr double c3[3] = {1.0, -0.5, -0.5};
	constexpr double c5[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
	                          0.30901699437494742410};
	constexpr double c7[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
	                          -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
	constexpr double c9[9] = {1.0, 0.76604444311897803520, 0.17364817766693034885, -0.5, -0.93969262078590838405,
	                          -0.93969262078590838405, -0.5, 0.17364817766693034885, 0.76604444311897803520};
	return P == 3 ? c3[j % 3] : P == 5 ? c5[j % 5] : P == 7 ? c7[j % 7] : c9[j % 9];
}
template <int P>
__device__ __forceinline__ constexpr double roots(int j) {
	constexpr double s3[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
	constexpr double s5[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
	                          -0.95105651629515357212};
	constexpr double s7[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048,
	                          -0.43388373911755812048, -0.97492791218182360702, -0.78183148246802980871};
	constexpr double s9[9] = {0.0, 0.64278760968653932632, 0.98480775301220805937, 0.86602540378443864676,
	                          0.34202014332566873304, -0.34202014332566873304, -0.86602540378443864676,
	                          -0.98480775301220805937, -0.64278760968653932632};
	return P == 3 ? s3[j % 3] : P == 5 ? s5[j % 5] : P == 7 ? s7[j % 7] : s9[j % 9];
}

// Odd prime P: with t_j = x_j + x_{P-j}, d_j = x_j - x_{P-j} (j = 1 ... (P-1)/2),
// y_k, y_{P-k} = (x_0 + sum c_{jk} t_j) +- SIGN i sum s_{jk} d_j.
template <int P, int SIGN>
__device__ __forceinline__ void dft_prime(double2 v[P]) {
	constexpr int H = (P - 1) / 2;
	double2 t[H], d[H], y0 = v[0];
#pragma unroll
	for (int j = 0; j < H; ++j) {
		t[j] = cadd(v[j + 1], v[P - 1 - j]);
		d[j] = csub(v[j + 1], v[P - 1 - j]);
		y0 = cadd(y0, t[j]);
	}
	const double2 x0 = v[0];
	v[0] = y0;
#pragma unroll
	for (int k = 1; k <= H; ++k) {
		double2 m = x0, n = make_double2(0.0, 0.0);
#pragma unroll
		for (int j = 1; j <= H; ++j) {
			const double c = rootc<P>(j * k), s = SIGN * roots<P>(j * k);
			m = make_double2(fma(c, t[j - 1].x, m.x), fma(c, t[j - 1].y, m.y));
			n = j == 1 ? make_double2(s * d[0].x, s * d[0].y)
			           : make_double2(fma(s, d[j - 1].x, n.x), fma(s, d[j - 1].y, n.y));
		}
		v[k] = make_double2(m.x - n.y, m.y + n.x);
		v[P - k] = make_double2(m.x + n.y, m.y - n.x);
	}
}

template <int P, int SIGN>
__device__ __forceinline__ void dft_nat(double2 v[P]);

// P = A B coprime: x at (B i + A j) mod P, X_k at the k with k = k1 mod A, k2 mod B.
template <int A, int B, int SIGN>
__device__ __forceinline__ void dft_coprime(double2 v[A * B]) {
	constexpr int P = A * B;
	double2 g[B][A];
#pragma unroll
	for (int j = 0; j < B; ++j) {
#pragma unroll
		for (int i = 0; i < A; ++i) g[j][i] = v[(B * i + A * j) % P];
		dft_nat<A, SIGN>(g[j]);
	}
#pragma unroll
	for (int i = 0; i < A; ++i) {
		double2 w[B];
#pragma unroll
		for (int j = 0; j < B; ++j) w[j] = g[j][i];
		dft_nat<B, SIGN>(w);
#pragma unroll
		for (int k = 0; k < P; ++k)
			if (k % A == i) v[k] = w[k % B];
	}
}

template <int P, int SIGN>
__device__ __forceinline__ void dft_nat(double2 v[P]) {
	if constexpr (P == 2) dft_n2p<2, SIGN>(v);
	else if constexpr (P == 4) dft4<SIGN>(v[0], v[1], v[2], v[3]);
	else if constexpr (P == 3 || P == 5 || P == 7) dft_prime<P, SIGN>(v);
	else if constexpr (P == 8 || P == 16) {
		dft_n2p<P, SIGN>(v);
		double2 w[P];
#pragma unroll
		for (int k = 0; k < P; ++k) w[k] = v[perm<P>(k)];
#pragma unroll
		for (int k = 0; k < P; ++k) v[k] = w[k];
	} else if constexpr (P == 9) { // 3 x 3 around the twiddles W9^{b c}
		double2 g[3][3];
#pragma unroll
		for (int b = 0; b < 3; ++b) {
#pragma unroll
			for (int a = 0; a < 3; ++a) g[b][a] = v[3 * a + b];
			dft_prime<3, SIGN>(g[b]);
		}
#pragma unroll
		for (int c = 0; c < 3; ++c) {
			double2 w[3];
#pragma unroll
			for (int b = 0; b < 3; ++b)
				w[b] = b * c ? cmul(g[b][c], make_double2(rootc<9>(b * c), SIGN * roots<9>(b * c))) : g[b][c];
			dft_prime<3, SIGN>(w);
#pragma unroll
			for (int k = 0; k < 3; ++k) v[c + 3 * k] = w[k];
		}
	} else if constexpr (P == 6) dft_coprime<2, 3, SIGN>(v);
	else if constexpr (P == 10) dft_coprime<2, 5, SIGN>(v);
	else if constexpr (P == 12) dft_coprime<4, 3, SIGN>(v);
	else if constexpr (P == 14) dft_coprime<2, 7, SIGN>(v);
	else {
		static_assert(P == 15, "");
		dft_coprime<3, 5, SIGN>(v);
	}
}
