// Bluestein's chirp-z tables of the DNLS step and the energy pass (host side).
#include "nlc_internal.hpp"

#include <algorithm>
#include <cmath>
#include <utility>
#include <vector>

namespace nlc {
namespace {

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
	if (n < 2 || pow2(n) || smooth_length(n)) return 0;
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

} // namespace nlc
