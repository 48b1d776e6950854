// Shared pieces of the register-resident step kernels (wave and workgroup
// forms): the Toda exp table, DPP / ds_bpermute lane moves and the FPUT / Toda
// bond terms.  Included inside namespace nlc { namespace { ... } } by
// nlc_step_wave.inl and nlc_step_group.inl, once per translation unit.
__constant__ double kExp2Tab[kExpTabSize] = NLC_EXP2_TABLE;

// Toda kernels: copy the exp table into LDS (every thread of the workgroup
// reaches the barrier).
template <int MODEL>
__device__ __forceinline__ void load_exp_table(double *lds) {
	if constexpr (MODEL == TODA) {
		for (uint32_t i = threadIdx.x; i < uint32_t(kExpTabSize); i += blockDim.x) lds[i] = kExp2Tab[i];
		__syncthreads();
	}
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
	const int lo = __double2loint(v), hi = __double2hiint(v);
	// every control used here reads a valid lane, so bound_ctrl never applies
	const int rlo = __builtin_amdgcn_mov_dpp(lo, CTRL, 0xF, 0xF, true);
	const int rhi = __builtin_amdgcn_mov_dpp(hi, CTRL, 0xF, 0xF, true);
	return __hiloint2double(rhi, rlo);
}

__device__ __forceinline__ double bperm_f64(double v, int src_lane) {
	const int addr = src_lane << 2;
	const int lo = __builtin_amdgcn_ds_bpermute(addr, __double2loint(v));
	const int hi = __builtin_amdgcn_ds_bpermute(addr, __double2hiint(v));
	return __hiloint2double(hi, lo);
}

// DPP controls (GFX9 encoding): wave_rol:1 = 0x134, wave_ror:1 = 0x13C,
// row_ror:n = 0x120+n, quad_perm = 8-bit lane selector.
constexpr int kWaveRol1 = 0x134;
constexpr int kWaveRor1 = 0x13C;
constexpr int kRowRor1 = 0x121;
constexpr int kRowRor15 = 0x12F;
constexpr int kQuadLeft = (3 << 0) | (0 << 2) | (1 << 4) | (2 << 6);  // lane i <- lane (i-1)&3
constexpr int kQuadRight = (1 << 0) | (2 << 2) | (3 << 4) | (0 << 6); // lane i <- lane (i+1)&3
constexpr int kQuadSwap = (1 << 0) | (0 << 2) | (3 << 4) | (2 << 6);  // lane i <- lane i^1

// Value held by the lane on the left (lane-1 within the chain's L-lane ring).
template <int L>
__device__ __forceinline__ double from_left(double v, int lane) {
	if constexpr (L == 1) return v;
	else if constexpr (L == 2) return dpp_f64<kQuadSwap>(v);
	else if constexpr (L == 4) return dpp_f64<kQuadLeft>(v);
	else if constexpr (L == 16) return dpp_f64<kRowRor1>(v);
	else if constexpr (L == 64) return dpp_f64<kWaveRor1>(v);
	else return bperm_f64(v, (lane & ~(L - 1)) | ((lane - 1) & (L - 1)));
}

// Value held by the lane on the right (lane+1 within the ring).
template <int L>
__device__ __forceinline__ double from_right(double v, int lane) {
	if constexpr (L == 1) return v;
	else if constexpr (L == 2) return dpp_f64<kQuadSwap>(v);
	else if constexpr (L == 4) return dpp_f64<kQuadRight>(v);
	else if constexpr (L == 16) return dpp_f64<kRowRor15>(v);
	else if constexpr (L == 64) return dpp_f64<kWaveRol1>(v);
	else return bperm_f64(v, (lane & ~(L - 1)) | ((lane + 1) & (L - 1)));
}

// The same moves for FP32 values (the FP32-compensated kernels).
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
	return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}

template <int L>
__device__ __forceinline__ float from_left(float v, int lane) {
	if constexpr (L == 1) return v;
	else if constexpr (L == 2) return dpp_f32<kQuadSwap>(v);
	else if constexpr (L == 4) return dpp_f32<kQuadLeft>(v);
	else if constexpr (L == 16) return dpp_f32<kRowRor1>(v);
	else if constexpr (L == 64) return dpp_f32<kWaveRor1>(v);
	else
		return __int_as_float(__builtin_amdgcn_ds_bpermute(((lane & ~(L - 1)) | ((lane - 1) & (L - 1))) << 2,
		                                                   __float_as_int(v)));
}

template <int L>
__device__ __forceinline__ float from_right(float v, int lane) {
	if constexpr (L == 1) return v;
	else if constexpr (L == 2) return dpp_f32<kQuadSwap>(v);
	else if constexpr (L == 4) return dpp_f32<kQuadRight>(v);
	else if constexpr (L == 16) return dpp_f32<kRowRor15>(v);
	else if constexpr (L == 64) return dpp_f32<kWaveRol1>(v);
	else
		return __int_as_float(__builtin_amdgcn_ds_bpermute(((lane & ~(L - 1)) | ((lane + 1) & (L - 1))) << 2,
		                                                   __float_as_int(v)));
}

// Force of DNKG / dDNKG on a site with neighbours l, r and mass = m_x + 2:
// l + r - q (m_x + 2 + beta q^2) (DNKG_FPUT_Toda.cu:24-31, dDNKG.cu:17-19).
// kFormCubic works on sigma q with sigma = sqrt(beta), where the cubic
// coefficient is 1: one FMA for m + 2 + q^2 instead of a product and an FMA.
template <int FORM>
__device__ __forceinline__ double site_force(double l, double q, double r, double mass, const StepArgs &a) {
	const double t = (FORM == kFormCubic) ? fma(q, q, mass) : fma(a.beta, q * q, mass);
	return fma(-q, t, l + r);
}

// Bond force term of FPUT / Toda for the bond x = q_{i} - q_{i-1}; the force on
// site i is bond(x_{i+1}) - bond(x_i).
//   FPUT: V'(x) = x + alpha x^2 + beta x^3  (Horner), the same force as
//         (l+r-2c)(1+alpha(r-l)) + beta(d_r^3-d_l^3) of DNKG_FPUT_Toda.cu:33-50;
//         on sigma q, kFormCubic (alpha = 0, sigma = sqrt(beta)) is x + x^3 and
//         kFormQuad (beta = 0, sigma = alpha) is x + x^2;
//   Toda: e^{2 alpha x}, the force of DNKG_FPUT_Toda.cu:52-66 without its factor
//         1/(2 alpha), which the kick folds into its weight (the constant
//         -1/(2 alpha) of V' cancels in the difference), evaluated as
//         2^(x'/256) on the bond x' = v_i - v_{i-1} of v = (512 alpha/ln2) q,
//         table driven (fewest instructions), or for S >= 25 sites per lane
//         the table-free form, 2^x' on the bond of v = (2 alpha/ln2) q
//         (toda_unit): more accurate than the plain table form by a third, and
//         with the rounding errors of the entries carried along to match it the
//         table form is bound by two LDS reads per bond (2048 sites x 4096, 100
//         steps: 3.5 ms table-free, 3.7).
template <int MODEL, int S, int FORM>
__device__ __forceinline__ double bond_force(double x, const StepArgs &a, const double *etab) {
	if constexpr (MODEL == FPUT) {
		if constexpr (FORM == kFormCubic) return fma(x * x, x, x);
		else if constexpr (FORM == kFormQuad) return fma(x, x, x);
		else return x * fma(x, fma(a.beta, x, a.alpha), 1.0);
	} else if constexpr (S >= 25) return exp2_poly(x); // Toda: x = v_i - v_{i-1}
	else return exp2_256_tab(x, etab);
}

// Kicks of a lane's S Toda sites in runs of R bonds: the reductions and table
// reads of a run are issued before the polynomials of the run before it, so the
// reads' latency passes behind 9 R instructions also where a SIMD has one wave.
// The empty asm statements (no instruction) hold that order: the next run's
// reductions come before this run's polynomials, and the run after it starts
// from here.  Without them the scheduler starts every site's read at once
// (196 VGPRs for 16 sites, two waves per SIMD, 125 and four with them; 256 and
// spills in the workgroup form) or, held to fewer registers, waits for each
// read in turn.
// R = 4 in the wave kernels; 2 in the workgroup kernels, which hold the halos
// too (8192 sites x 512: 1.89 ms, with R = 4 2.05 ms: 3 waves per SIMD).
// 100 steps, without and with: 1024 x 8192 3.03 and 2.87 ms, 500 x 8192 1.76
// and 1.60, 1500 x 4096 2.99 and 2.24, 3000 x 2048 6.8 and 3.0, 12000 x 256 2.90
// and 1.46 (the workgroup form spilled).
// For 8 to 24 sites per lane: with fewer a run is the whole lane, from 25 on the
// bonds are table-free.
// bl: the lane's first bond; bs: the right bond of its last real site.
template <int S>
constexpr bool toda_in_runs() { return S >= 8 && S < 25; }

template <int R, int S, bool EXACT>
__device__ __forceinline__ void toda_kicks(double (&p)[S], double (&q)[S], double w, double bl, double bs, bool full,
                                           const double *etab) {
	Exp2Red d[2][R];
#pragma unroll
	for (int i = 0; i < R; ++i) d[0][i] = exp2_256_reduce(q[i + 1] - q[i], etab);
#pragma unroll
	for (int j = 0; j < S; j += R) {
		Exp2Red *const cur = d[(j / R) % 2], *const next = d[(j / R + 1) % 2];
#pragma unroll
		for (int i = 0; i < R; ++i)
			if (j + R + i < S - 1) next[i] = exp2_256_reduce(q[j + R + i + 1] - q[j + R + i], etab);
#pragma unroll
		for (int i = 0; i < R; ++i)
			if (j + i < S - 1) asm volatile("" : "+v"(cur[i].r));
#pragma unroll
		for (int i = 0; i < R; ++i) {
			if (j + i >= S) break;
			double br = bs;
			if (j + i < S - 1) br = exp2_256_finish(cur[i]);
			if (!EXACT && j + i == S - 2) br = full ? br : bs;
			p[j + i] = fma(w, br - bl, p[j + i]);
			bl = br;
		}
#pragma unroll
		for (int i = 0; i < R; ++i) {
			if (j + i < S) asm volatile("" : "+v"(p[j + i]));
			if (j + 2 * R + i < S) asm volatile("" : "+v"(q[j + 2 * R + i]));
		}
	}
}

// Unit of the Toda state in a kernel with S sites per lane, relative to v =
// (256 alpha/ln2) q: 2 for the table form (bond exponent in table steps of 1/256
// octave; 1, 1/128 octave, in the FP32-compensated kernels), 2^-7 for the
// table-free form's (2 alpha/ln2) q (octaves).  Scaling by a power of two is
// exact, so all hold the same trajectory.
template <int MODEL, int S, bool C32 = false>
__device__ __forceinline__ constexpr double toda_unit() {
	return MODEL != TODA ? 1.0 : S >= 25 ? 0x1p-7 : C32 ? 1.0 : 2.0;
}

// The state as the kernels hold it: sigma q and sigma p for the scaled forms
// (then sigma F(q) = F~(sigma q), so drift and kick weights stay as they
// are), v = sigma q with unscaled p for Toda (sigma = 256 alpha/ln2 times
// toda_unit), else q and p.  The way back multiplies by 1/sigma: a division
// would put its 10-instruction sequence between the stores of a lane, and the
// L2 then writes partly filled lines back (a third more HBM write traffic
// measured).
template <int MODEL, int FORM, int S, bool C32 = false>
__device__ __forceinline__ double2 to_registers(double2 v, const StepArgs &a) {
	if constexpr (MODEL == TODA) return make_double2((a.scale * toda_unit<MODEL, S, C32>()) * v.x, v.y);
	else if constexpr (FORM != kFormPlain) return make_double2(a.scale * v.x, a.scale * v.y);
	else return v;
}

template <int MODEL, int FORM, int S, bool C32 = false>
__device__ __forceinline__ double2 from_registers(double q, double p, const StepArgs &a) {
	if constexpr (MODEL == TODA) return make_double2(q * (a.inv_scale / toda_unit<MODEL, S, C32>()), p);
	else if constexpr (FORM != kFormPlain) return make_double2(q * a.inv_scale, p * a.inv_scale);
	else return make_double2(q, p);
}

