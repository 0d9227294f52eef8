// stab.hip -- the slice product with periodic FP64 stabilisation: log det and inverse of
// 1 + B_0 B_1 ... B_{nt-1} without forming the product's full dynamic range in one matrix.
//
// The product is kept as U diag(d) V (U orthogonal, d > 0 the column scales, V of O(1) entries) and
// grown by blocks of k slices, in the reference's order (slices nt-1 first, applied from the left,
// construct_M_hat organic_dense_matrix.c:256-258):
//     Y = B_lo ... B_hi U                  (the chain kernels, in the slice precision)
//     Z = Y diag(d) Pi                     (columns sorted by norm, largest first: pre-pivoting)
//     Z = Q R                              (FP64 Householder QR)
//     U <- Q,  d <- |diag R|,  V <- (diag(d)^{-1} R) Pi^T V
// Every block's dynamic range is that of k slices only, so an FP32 block loses nothing the FP64
// factorisation cannot hold.  At the end, with D_b = max(d, 1) and D_s = min(d, 1),
//     1 + U D V = U D_b X,   X = D_b^{-1} U^T + D_s V,
// so log|det(1 + U D V)| = sum log D_b + log|det X| (det U = +-1) and
//     (1 + U D V)^{-1} = X^{-1} D_b^{-1} U^T;
// X is well conditioned however wide d is, and X = Q R gives its determinant and
// X^{-1} C = R^{-1} (Q^T C) without row exchanges.
//
// The pre-pivoting is decided before the factorisation, so the QR needs no column exchanges and is
// blocked: panels of NB columns are factorised by one workgroup in registers, and every other
// column receives the panel's NB reflectors at once as I - V T V^T (compact WY) on the FP64 matrix
// cores, 16 columns per workgroup.  One launch per panel: workgroup 0 updates and factorises the
// next panel while the others update the columns behind it.  What bounds it is the chain of N
// dependent reflectors per block, 1.2 us each (two barriers, the reduction over the rows, a square
// root and two reciprocals); the products around it take a fifth of the time.
// N = 256, nt = 64, k = 8, one log det and inverse: 4.8 ms.  One workgroup for the whole matrix, which
// streamed it through one CU for every reflector, and a pivoted Gauss-Jordan for X took 55.2 ms.
#include "internal.h"

namespace ephmc {

typedef double st_v4d __attribute__((ext_vector_type(4)));

// log(d_c) + log|Y_c| of every column (logs: the scales may span far more than an FP64 square);
// one wave per column.  A NaN ranks as the largest key, so that the order stays a permutation.
template <typename R>
__global__ __launch_bounds__(256) void qr_key_kernel(const R *__restrict__ Y, const double *__restrict__ d, unsigned n,
		double *__restrict__ key)
{
	const unsigned c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if(c >= n) return;
	const R *y = Y + (size_t)c * n;
	double s = 0;
	for(unsigned r = lane; r < n; r += 64){ const double v = (double)y[r]; s = fma(v, v, s); }
#pragma unroll
	for(int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
	if(lane == 0){
		const double k = s > 0 ? log(d[c]) + 0.5 * log(s) : (s == 0 ? -HUGE_VAL : HUGE_VAL);
		key[c] = k == k ? k : HUGE_VAL;
	}
}

// Z = Y diag(d) Pi with the columns by key, largest first, ties by column index; one workgroup per
// source column.  perm[k] = source column of column k.
template <typename R>
__global__ __launch_bounds__(256) void qr_sort_kernel(const R *__restrict__ Y, const double *__restrict__ d,
		const double *__restrict__ key, unsigned n, double *__restrict__ z, int *__restrict__ perm)
{
	__shared__ unsigned cnt[4];
	const unsigned c = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const double kc = key[c];
	unsigned rank = 0;
	for(unsigned o = threadIdx.x; o < n; o += 256){
		const double ko = key[o];
		rank += (ko > kc || (ko == kc && o < c)) ? 1u : 0u;
	}
#pragma unroll
	for(int off = 32; off > 0; off >>= 1) rank += __shfl_xor(rank, off, 64);
	if(lane == 0) cnt[wave] = rank;
	__syncthreads();
	rank = cnt[0] + cnt[1] + cnt[2] + cnt[3];
	const double dc = d[c];
	for(unsigned r = threadIdx.x; r < n; r += 256) z[(size_t)rank * n + r] = dc * (double)Y[(size_t)c * n + r];
	if(threadIdx.x == 0) perm[rank] = (int)c;
}

// v + (v of lane ^ off), off = 8, 16 or 32, without LDS: a row rotation or the half-row / half-wave swaps
template <int OFF>
__device__ __forceinline__ double xor_sum(double v)
{
	const long long b = __double_as_longlong(v);
	const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
	static_assert(OFF == 8 || OFF == 16 || OFF == 32, "");
	if constexpr(OFF == 8){
		const unsigned l2 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)lo, 0x128, 0xf, 0xf, false);
		const unsigned h2 = (unsigned)__builtin_amdgcn_update_dpp(0, (int)hi, 0x128, 0xf, 0xf, false);
		return v + __longlong_as_double(((long long)h2 << 32) | l2);
	}else if constexpr(OFF == 16){
		const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false), h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
		return __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
	}else{
		const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false), h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
		return __longlong_as_double(((long long)h[0] << 32) | l[0]) + __longlong_as_double(((long long)h[1] << 32) | l[1]);
	}
}

// Doubles of LDS that apply_block uses.
template <int NB, int CB>
constexpr int wy_lds(){ return 8 * NB * 16 + NB * (NB + 1) + 2 * CB * NB * 17; }

// zt <- (1 - V T V^T) zt, or with T^T (trans), for ncol <= 16 CB columns of zt (column-major, leading
// dimension n).  V of the panel at column j0: vp[i ldv + r], zero outside its support and past row
// n, so its loads carry no conditions.  All BT threads of the workgroup.
// Phase 1, W^T = zt^T V: up to eight waves, shared out over the 16-column blocks, take 64-row blocks
// in turn and accumulate all NB columns; the waves' sums meet in LDS.  Phase 2, T W: T from LDS.
// Phase 3, zt -= V (T W): 64-row blocks over all waves, transposed so that 16 lanes hold 16
// consecutive rows and the loads and stores coalesce.  A block's loads are all issued before its
// products: the panel comes from another workgroup's stores, so every dependent round of loads
// would cost most of a microsecond.
template <int NB, int BT, int CB>
__device__ __forceinline__ void apply_block(const double *__restrict__ vp, unsigned ldv, unsigned n, unsigned j0,
		const double *__restrict__ tm, bool trans, double *zt, unsigned ncol, double *sm)
{
	constexpr int NW = BT / 64, NW1 = (NW < 8 ? NW : 8) / CB;
	const unsigned tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m16 = lane & 15, k4 = lane >> 4;
	double *part = sm, *tl = part + 8 * NB * 16, *ws = tl + NB * (NB + 1), *w2 = ws + CB * NB * 17;
	for(unsigned e = tid; e < NB * NB; e += BT){          // tl[k][i]: the factor of entry k in sum i
		const unsigned r = e / NB, c = e % NB;
		tl[trans ? r * (NB + 1) + c : c * (NB + 1) + r] = tm[e];
	}
	if(wave < NW1 * CB){
		const unsigned cb = wave / NW1, w1 = wave % NW1;
		const double *zp = zt + (size_t)min(16 * cb + m16, ncol - 1) * n;
		st_v4d acc[NB / 16];
#pragma unroll
		for(int ib = 0; ib < NB / 16; ib++) acc[ib] = st_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
		for(unsigned r0 = j0 + 64 * w1; r0 < n; r0 += 64 * NW1){
			double zv[16], vv[NB / 16][16];
			const double *v0 = vp + (size_t)m16 * ldv + r0 + k4;
#pragma unroll
			for(int q = 0; q < 16; q++){
				zv[q] = zp[min(r0 + 4 * q + k4, n - 1)];
#pragma unroll
				for(int ib = 0; ib < NB / 16; ib++) vv[ib][q] = (v0 + (size_t)(16 * ib) * ldv)[4 * q];
			}
#pragma unroll
			for(int q = 0; q < 16; q++)
#pragma unroll
				for(int ib = 0; ib < NB / 16; ib++)
					acc[ib] = __builtin_amdgcn_mfma_f64_16x16x4f64(zv[q], vv[ib][q], acc[ib], 0, 0, 0);
		}
#pragma unroll
		for(int ib = 0; ib < NB / 16; ib++)
#pragma unroll
			for(int e = 0; e < 4; e++) part[(wave * NB + 16 * ib + m16) * 16 + 4 * e + k4] = acc[ib][e];
	}
	__syncthreads();
	for(unsigned e = tid; e < CB * NB * 16; e += BT){
		const unsigned cb = e / (NB * 16), f = e % (NB * 16);
		double s = part[cb * NW1 * NB * 16 + f];
#pragma unroll
		for(int w = 1; w < NW1; w++) s += part[(cb * NW1 + w) * NB * 16 + f];
		ws[(e >> 4) * 17 + (e & 15)] = s;
	}
	__syncthreads();
	for(unsigned e = tid; e < CB * NB * 16; e += BT){
		const unsigned cb = e / (NB * 16), i = (e >> 4) % NB, col = e & 15;
		double s0 = 0, s1 = 0;
#pragma unroll 8
		for(int k = 0; k < NB; k += 2){
			s0 = fma(tl[k * (NB + 1) + i], ws[(cb * NB + k) * 17 + col], s0);
			s1 = fma(tl[(k + 1) * (NB + 1) + i], ws[(cb * NB + k + 1) * 17 + col], s1);
		}
		w2[(e >> 4) * 17 + col] = -(s0 + s1);
	}
	__syncthreads();
#pragma unroll 1
	for(unsigned r0 = j0 + 64 * wave; r0 < n; r0 += 64 * NW){
		st_v4d acc[4][CB];
		double vv[NB / 4][4];
		const double *v0 = vp + (size_t)k4 * ldv + r0 + m16;
#pragma unroll
		for(int b = 0; b < 4; b++){
#pragma unroll
			for(int kb = 0; kb < NB / 4; kb++) vv[kb][b] = (v0 + (size_t)(4 * kb) * ldv)[16 * b];
#pragma unroll
			for(int cb = 0; cb < CB; cb++)
#pragma unroll
				for(int e = 0; e < 4; e++)
					acc[b][cb][e] = zt[(size_t)min(16 * cb + 4 * e + k4, ncol - 1) * n + min(r0 + 16 * b + m16, n - 1)];
		}
#pragma unroll
		for(int kb = 0; kb < NB / 4; kb++)
#pragma unroll
			for(int cb = 0; cb < CB; cb++){
				const double w = w2[(cb * NB + 4 * kb + k4) * 17 + m16];
#pragma unroll
				for(int b = 0; b < 4; b++)
					acc[b][cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(w, vv[kb][b], acc[b][cb], 0, 0, 0);
			}
#pragma unroll
		for(int b = 0; b < 4; b++)
#pragma unroll
			for(int cb = 0; cb < CB; cb++)
#pragma unroll
				for(int e = 0; e < 4; e++){
					const unsigned col = 16 * cb + 4 * e + k4, r = r0 + 16 * b + m16;
					if(col < ncol && r < n) zt[(size_t)col * n + r] = acc[b][cb][e];
				}
	}
	__syncthreads();
}

// t (NB x NB in LDS, leading dimension NB + 1, diagonal given, all else to be formed) <- the upper
// triangular matrix with t_12 = -t_11 s_12 t_22 for every pair of neighbouring diagonal blocks of
// size 1, 2, 4, ..: the inverse of an upper triangular s with t_ii = 1 / s_ii, and the T factor of
// NB reflectors with t_ii = t_i and s = V^T V above the diagonal.  s(i, k) = sp[k (NB + 1) + i].
// Ten short parallel products in place of a chain of NB dependent rows.
template <int NB, int BT>
__device__ __forceinline__ void upper_from_diagonal(const double *sp, double *t, double *tmp)
{
	constexpr int LD = NB + 1;
#pragma unroll 1
	for(int lb = 0; (1 << lb) < NB; lb++){
		const int b = 1 << lb;
		for(int e = threadIdx.x; e < (NB / 2) << lb; e += BT){
			const int j0 = (e >> (2 * lb)) << (lb + 1), i = j0 + ((e >> lb) & (b - 1)), j = j0 + b + (e & (b - 1));
			double s = 0;
#pragma unroll 4
			for(int k = j0 + b; k <= j; k++) s = fma(sp[k * LD + i], t[k * LD + j], s);
			tmp[i * LD + j] = s;
		}
		__syncthreads();
		for(int e = threadIdx.x; e < (NB / 2) << lb; e += BT){
			const int j0 = (e >> (2 * lb)) << (lb + 1), i = j0 + ((e >> lb) & (b - 1)), j = j0 + b + (e & (b - 1));
			double s = 0;
#pragma unroll 4
			for(int k = i; k < j0 + b; k++) s = fma(t[i * LD + k], tmp[k * LD + j], s);
			t[i * LD + j] = -s;
		}
		__syncthreads();
	}
}

// 1/x and sqrt(x) for x > 0 from the hardware estimates with Newton steps (within an ulp or so; the
// reflectors need no more, and the exact forms are most of a step's dependent chain)
__device__ __forceinline__ double st_rcp(double x)
{
	double r = __builtin_amdgcn_rcp(x);
	r = fma(r, fma(-x, r, 1.0), r);
	return fma(r, fma(-x, r, 1.0), r);
}

__device__ __forceinline__ double st_sqrt(double x)
{
	double y = __builtin_amdgcn_rsq(x);
	y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
	const double g = x * y;
	return fma(0.5 * y, fma(-g, g, x), g);
}

// Householder factorisation of the panel of nb <= NB columns at column j0 of z, rows j0.. (all BT
// threads).  Thread (c4 = tid % (NB / 4), g = tid / (NB / 4)) holds the columns 4 c4 .. 4 c4 + 3 at
// the RPT rows
//     rr = (q / 2) 2 G + 2 g + q % 2,  G = 4 BT / NB  (relative to j0, G RPT >= n - j0),
// so a reflector's products need no data but the reflector itself, read from LDS once for four
// columns (one column per thread reads LDS four times as much and took 2.2 us per reflector).
// Step jj publishes column jj below the diagonal and row jj; every thread forms its rows' share of
// s_c = sum_{r > jj} x_r a_rc for its columns, and the sums over g give, for every column at once,
//     w_c = v_jj . a_c = a_jj,c + s_c / (alpha - beta):
// the update of the columns c > jj, the squared norm at c = jj, and for c < jj the entry v_c . v_jj
// from which T follows.  Two barriers per step.  Four steps are unrolled, so that every
// choice of a column or row is a register named in the code; all NB unrolled would be executed once
// per launch and wait for its instruction fetches, and one step with the choices made by selects
// takes 2.5 us against 1.2 us.  R goes back to z, the reflectors to vp (leading dimension ldv), T to tm.
template <int NB, int BT, int RPT>
__device__ __forceinline__ void factor_panel(double *__restrict__ z, unsigned n, unsigned j0, unsigned nb,
		double *__restrict__ vp, unsigned ldv, double *__restrict__ tm, int *__restrict__ nref, bool first, double *sm)
{
	constexpr int NC = NB / 4, G = BT / NC, NW = BT / 64, LX = RPT + 2, LD = NB + 1;
	static_assert(2 * G >= NB, "row jj sits in q = jj % 2");
	const int tid = threadIdx.x, c4 = tid % NC, g = tid / NC, lane = tid & 63, wave = tid >> 6;
	double *xs = sm, *zs = xs + 2 * G * LX, *part = zs + 2 * NB, *gm = part + NW * NB, *tl = gm + NB * LD, *tmp = tl + NB * LD;
	double a[4][RPT];
	const int m = (int)(n - j0);
#pragma unroll
	for(int k = 0; k < 4; k++)
#pragma unroll
		for(int q = 0; q < RPT; q++){
			const int rr = (q >> 1) * 2 * G + 2 * g + (q & 1);
			a[k][q] = z[(size_t)min(j0 + 4 * c4 + k, n - 1) * n + min(j0 + rr, n - 1)];
			if(4 * c4 + k >= (int)nb || rr >= m) a[k][q] = 0.0;
		}
	// T, and V^T V: the sums for T run over all NB columns, of which a panel of nb < NB forms nb
	for(int e = tid; e < 2 * NB * LD; e += BT) gm[e] = 0.0;
	int refl = 0;
#pragma unroll 1
	for(int jq = 0; jq < NC; jq++)
#pragma unroll
	for(int kj = 0; kj < 4; kj++){
		const int jj = 4 * jq + kj, par = kj & 1;
		if(jj >= (int)nb) break;
		const bool own = g == (jj >> 1);                           // holds row jj, in a[.][par]
		double *xp = xs + (par * G + g) * LX, *zrow = zs + par * NB;
		if(c4 == jq){
#pragma unroll
			for(int q = 0; q < RPT; q++){
				const int rr = (q >> 1) * 2 * G + 2 * g + (q & 1);
				xp[q] = rr > jj ? a[kj][q] : 0.0;
			}
		}
		if(own)
#pragma unroll
			for(int k = 0; k < 4; k++) zrow[4 * c4 + k] = a[k][par];
		__syncthreads();
		double x[RPT], s[4] = {0, 0, 0, 0};
#pragma unroll
		for(int q = 0; q < RPT; q++) x[q] = xp[q];
#pragma unroll
		for(int q = 0; q < RPT; q++)
#pragma unroll
			for(int k = 0; k < 4; k++) s[k] = fma(x[q], a[k][q], s[k]);
#pragma unroll
		for(int k = 0; k < 4; k++){
			if constexpr(NC == 4) s[k] += __shfl_xor(s[k], 4, 64);
			s[k] = xor_sum<32>(xor_sum<16>(xor_sum<8>(s[k])));
		}
		if(lane < NC)
#pragma unroll
			for(int k = 0; k < 4; k++) part[wave * NB + 4 * lane + k] = s[k];
		__syncthreads();
		double sig = 0, sc[4] = {0, 0, 0, 0};
#pragma unroll
		for(int w = 0; w < NW; w++){
			sig += part[w * NB + jj];
#pragma unroll
			for(int k = 0; k < 4; k++) sc[k] += part[w * NB + 4 * c4 + k];
		}
		const double alpha = zrow[jj];
		double t = 0, scale = 0, beta = alpha;
		if(!(sig == 0)){                                           // (a NaN column runs through as NaN)
			const double nrm = st_sqrt(fma(alpha, alpha, sig)), rn = st_rcp(nrm);
			beta = alpha >= 0 ? -nrm : nrm;
			scale = st_rcp(alpha - beta);
			t = (beta - alpha) * (alpha >= 0 ? -rn : rn);
			refl++;
		}
		if(tid == 0) tl[jj * (LD + 1)] = t;
		if(own) x[par] = alpha - beta;                             // v_jj = 1 = x scale
		const double tsc = t * scale;
#pragma unroll
		for(int k = 0; k < 4; k++){
			const double w = fma(scale, sc[k], zrow[4 * c4 + k]);
			if(g == 0 && 4 * c4 + k < jj) gm[jj * LD + 4 * c4 + k] = w;
			const double tw = 4 * c4 + k > jj ? tsc * w : 0.0;
#pragma unroll
			for(int q = 0; q < RPT; q++) a[k][q] = fma(-tw, x[q], a[k][q]);
		}
		if(c4 == jq){
#pragma unroll
			for(int q = 0; q < RPT; q++){
				const int rr = (q >> 1) * 2 * G + 2 * g + (q & 1);
				a[kj][q] = rr > jj ? x[q] * scale : (rr == jj ? beta : a[kj][q]);
			}
		}
	}
#pragma unroll
	for(int k = 0; k < 4; k++){
		const int cc = 4 * c4 + k;
		if(cc >= (int)nb) break;
#pragma unroll
		for(int q = 0; q < RPT; q += 2){
			const int rr = q * G + 2 * g;                          // rows rr and rr + 1
			if(rr >= m) break;
			if(q * G < NB){
				if(rr <= cc) z[(size_t)(j0 + cc) * n + j0 + rr] = a[k][q];
				if(rr + 1 <= cc && rr + 1 < m) z[(size_t)(j0 + cc) * n + j0 + rr + 1] = a[k][q + 1];
			}
			double2 v;
			v.x = rr > cc ? a[k][q] : (rr == cc ? 1.0 : 0.0);
			v.y = rr + 1 > cc ? a[k][q + 1] : (rr + 1 == cc ? 1.0 : 0.0);     // (zero past the last row)
			*(double2 *)(vp + (size_t)cc * ldv + j0 + rr) = v;     // j0, ldv and rr are even
		}
	}
	if(tid == 0) *nref = (first ? 0 : *nref) + refl;
	__syncthreads();
	// T: T_jj = t_j, V^T V = gm (both zero past nb: those rows and columns of T stay zero)
	upper_from_diagonal<NB, BT>(gm, tl, tmp);
	for(int e = tid; e < NB * NB; e += BT) tm[e] = tl[(e / NB) * LD + e % NB];
}

template <int NB, int BT, int RPT>
constexpr int qr_lds()
{
	constexpr int G = 4 * BT / NB, f = 2 * G * (RPT + 2) + 2 * NB + (BT / 64) * NB + 3 * NB * (NB + 1);
	return f > wy_lds<NB, NB / 16>() ? f : wy_lds<NB, NB / 16>();
}

// Step p of the blocked QR of z (p = -1 first): workgroup 0 applies panel p to the columns of panel
// p + 1 and factorises it, workgroup b >= 1 applies panel p to 16 of the columns behind it.
template <int NB, int BT, int RPT>
__global__ __launch_bounds__(BT) void qr_step_kernel(double *__restrict__ z, unsigned n, int p, double *__restrict__ vm,
		unsigned ldv, double *__restrict__ tm, int *__restrict__ nref)
{
	__shared__ __align__(16) double sm[qr_lds<NB, BT, RPT>()];
	const unsigned j1 = (unsigned)(p + 1) * NB, j0 = p < 0 ? 0 : (unsigned)p * NB;
	const double *tp = tm + (size_t)j0 * NB, *vp = vm + (size_t)j0 * ldv;
	if(blockIdx.x > 0){
		const unsigned c0 = j1 + NB + 16 * (blockIdx.x - 1);
		apply_block<NB, BT, 1>(vp, ldv, n, j0, tp, true, z + (size_t)c0 * n, min(16u, n - c0), sm);
		return;
	}
	const unsigned nb = min((unsigned)NB, n - j1);
	if(p >= 0) apply_block<NB, BT, NB / 16>(vp, ldv, n, j0, tp, true, z + (size_t)j1 * n, nb, sm);
	factor_panel<NB, BT, RPT>(z, n, j1, nb, vm + (size_t)j1 * ldv, ldv, tm + (size_t)j1 * NB, nref, p < 0, sm);
}

// q = Q = H_0 H_1 ... (column-major), 16 columns per workgroup: the panels are applied to the
// identity, last first; those past the tile's last column leave it as it is.
template <int NB>
__global__ __launch_bounds__(256) void qr_form_q_kernel(const double *__restrict__ vm, unsigned ldv, const double *__restrict__ tm,
		unsigned n, double *__restrict__ q)
{
	__shared__ __align__(16) double sm[wy_lds<NB, 1>()];
	const unsigned c0 = blockIdx.x * 16, nc = min(16u, n - c0);
	double *qt = q + (size_t)c0 * n;
	for(unsigned e = threadIdx.x; e < nc * n; e += 256) qt[e] = e % n == c0 + e / n ? 1.0 : 0.0;
	__syncthreads();
	for(int p = (int)((c0 + nc - 1) / NB); p >= 0; p--){
		const unsigned j0 = (unsigned)p * NB;
		apply_block<NB, 256, 1>(vm + (size_t)j0 * ldv, ldv, n, j0, tm + (size_t)j0 * NB, false, qt, nc, sm);
	}
}

// v_new = (diag(|R_ii|)^{-1} R) Pi^T v and d_new[i] = |R_ii|: 32 x 32 tiles, one 16 x 16 quadrant
// per wave on the matrix cores, transposed (16 lanes on 16 consecutive rows of R and v_new); the
// columns of R left of the tile's first row are skipped.
__global__ __launch_bounds__(256) void qr_update_v_kernel(const double *__restrict__ zr, const int *__restrict__ perm,
		unsigned n, const double *__restrict__ v, double *__restrict__ v_new, double *__restrict__ d_new)
{
	extern __shared__ int pl[];
	const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6, m16 = lane & 15, k4 = lane >> 4;
	const unsigned r0 = blockIdx.x * 32 + 16 * (wave & 1), c0 = blockIdx.y * 32 + 16 * (wave >> 1);
	for(unsigned k = threadIdx.x; k < n; k += 256) pl[k] = perm[k];
	__syncthreads();
	if(r0 >= n || c0 >= n) return;
	const unsigned row = r0 + m16, zrow = min(row, n - 1);
	const double *vc = v + (size_t)min(c0 + m16, n - 1) * n;
	st_v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
	for(unsigned k0 = r0; k0 < n; k0 += 64){
		double vv[16], rv[16];
#pragma unroll
		for(int q = 0; q < 16; q++){
			const unsigned k = k0 + 4 * q + k4, ks = min(k, n - 1);
			vv[q] = vc[pl[ks]];
			rv[q] = zr[(size_t)ks * n + zrow];
			if(k >= n) vv[q] = 0.0;
			if(k >= n || k < row) rv[q] = 0.0;
		}
#pragma unroll
		for(int q = 0; q < 16; q++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(vv[q], rv[q], acc, 0, 0, 0);
	}
	if(row >= n) return;
	const double rd = fabs(zr[(size_t)row * n + row]);
	if(blockIdx.y == 0 && wave < 2 && k4 == 0) d_new[row] = rd;
#pragma unroll
	for(int e = 0; e < 4; e++){
		const unsigned col = c0 + 4 * e + k4;
		if(col < n) v_new[(size_t)col * n + row] = acc[e] / rd;
	}
}

// X = D_b^{-1} U^T + D_s V (column-major), D_b = max(d, 1), D_s = min(d, 1)
__global__ __launch_bounds__(256) void stab_x_kernel(const double *__restrict__ u, const double *__restrict__ v,
		const double *__restrict__ d, unsigned n, double *__restrict__ x)
{
	__shared__ double tile[32][33];
	const unsigned bx = blockIdx.x * 32, by = blockIdx.y * 32;
	const unsigned tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
	// tile of U: rows bx.., columns by..  ->  transposed into X rows by.., columns bx..
	for(unsigned r = ty; r < 32; r += 8){
		const unsigned col = by + r, row = bx + tx;
		if(col < n && row < n) tile[r][tx] = u[(size_t)col * n + row];
	}
	__syncthreads();
	for(unsigned r = ty; r < 32; r += 8){
		const unsigned col = bx + r, row = by + tx;     // X(row, col) = U(col, row) / Db_row + Ds_row V(row, col)
		if(col < n && row < n){
			const double dr = d[row];
			const double db = dr > 1 ? dr : 1.0, ds = dr < 1 ? dr : 1.0;
			x[(size_t)col * n + row] = tile[tx][r] / db + ds * v[(size_t)col * n + row];
		}
	}
}

// Inverses of the diagonal blocks of R (upper triangular, row-major NB x NB, the last block padded
// with the identity), one workgroup each.
template <int NB>
__global__ __launch_bounds__(256) void tri_inverse_kernel(const double *__restrict__ zr, unsigned n, double *__restrict__ rinv)
{
	constexpr int LD = NB + 1;
	__shared__ double rs[NB * LD], t[NB * LD], tmp[NB * LD];
	const unsigned j0 = blockIdx.x * NB;
	for(unsigned e = threadIdx.x; e < NB * NB; e += 256){
		const unsigned k = e / NB, i = e % NB;              // R(j0 + i, j0 + k)
		const double v = zr[(size_t)min(j0 + k, n - 1) * n + min(j0 + i, n - 1)];
		rs[k * LD + i] = j0 + k < n ? v : 0.0;
		t[k * LD + i] = i == k ? (j0 + k < n ? 1.0 / v : 1.0) : 0.0;
	}
	__syncthreads();
	upper_from_diagonal<NB, 256>(rs, t, tmp);
	for(unsigned e = threadIdx.x; e < NB * NB; e += 256) rinv[(size_t)j0 * NB + e] = t[(e / NB) * LD + e % NB];
}

// minv = X^{-1} D_b^{-1} U^T with X = Q R factorised in zr, vm, tm, rinv: 16 columns per workgroup.
// C = Q^T (D_b^{-1} U^T) panel by panel, then R Y = C from the last block row up:
// Y_p = R_pp^{-1} C_p, C_above -= R_above,p Y_p.  An exactly zero R_ii (singular X): NaN.
template <int NB>
__global__ __launch_bounds__(256) void stab_solve_kernel(const double *__restrict__ zr, const double *__restrict__ vm, unsigned ldv, const double *__restrict__ tm,
		const double *__restrict__ rinv, const double *__restrict__ u, const double *__restrict__ d, unsigned n,
		double *__restrict__ minv)
{
	__shared__ __align__(16) double sm[wy_lds<NB, 1>()];
	const unsigned tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m16 = lane & 15, k4 = lane >> 4;
	const unsigned c0 = blockIdx.x * 16, nc = min(16u, n - c0);
	double *ct = minv + (size_t)c0 * n;
	int zero = 0;
	for(unsigned i = tid; i < n; i += 256) zero |= zr[(size_t)i * n + i] == 0;
	if(__syncthreads_or(zero)){
		for(unsigned e = tid; e < nc * n; e += 256) ct[e] = __longlong_as_double(0x7ff8000000000000LL);
		return;
	}
	for(unsigned e = tid; e < 16 * n; e += 256){
		const unsigned cc = e & 15, r = e >> 4;
		if(cc < nc) ct[(size_t)cc * n + r] = u[(size_t)r * n + c0 + cc] / (d[r] > 1 ? d[r] : 1.0);
	}
	__syncthreads();
	const int np = (int)((n + NB - 1) / NB);
	for(int p = 0; p < np; p++){
		const unsigned j0 = (unsigned)p * NB;
		apply_block<NB, 256, 1>(vm + (size_t)j0 * ldv, ldv, n, j0, tm + (size_t)j0 * NB, true, ct, nc, sm);
	}
	double *cs = sm, *ys = sm + NB * 17;
	for(int p = np - 1; p >= 0; p--){
		const unsigned j0 = (unsigned)p * NB, nb = min((unsigned)NB, n - j0);
		for(unsigned e = tid; e < NB * 16; e += 256){
			const unsigned cc = e / NB, i = e % NB;
			cs[i * 17 + cc] = (cc < nc && i < nb) ? ct[(size_t)cc * n + j0 + i] : 0.0;
		}
		__syncthreads();
		for(unsigned e = tid; e < NB * 16; e += 256){
			const unsigned cc = e / NB, i = e % NB;
			double s = 0;
			for(int k = 0; k < NB; k++) s = fma(rinv[(size_t)p * NB * NB + i * NB + k], cs[k * 17 + cc], s);
			ys[i * 17 + cc] = -s;
			if(cc < nc && i < nb) ct[(size_t)cc * n + j0 + i] = s;
		}
		__syncthreads();
		for(unsigned r0 = 16 * wave; r0 < j0; r0 += 64){
			const unsigned r = r0 + m16;                    // j0 is a multiple of 16
			st_v4d acc;
			double rv[NB / 4];
#pragma unroll
			for(int e = 0; e < 4; e++) acc[e] = 4 * e + k4 < nc ? ct[(size_t)(4 * e + k4) * n + r] : 0.0;
#pragma unroll
			for(int kb = 0; kb < NB / 4; kb++){
				const unsigned k = 4 * kb + k4;
				rv[kb] = k < nb ? zr[(size_t)(j0 + k) * n + r] : 0.0;
			}
#pragma unroll
			for(int kb = 0; kb < NB / 4; kb++)
				acc = __builtin_amdgcn_mfma_f64_16x16x4f64(ys[(4 * kb + k4) * 17 + m16], rv[kb], acc, 0, 0, 0);
#pragma unroll
			for(int e = 0; e < 4; e++)
				if(4 * e + k4 < nc) ct[(size_t)(4 * e + k4) * n + r] = acc[e];
		}
		__syncthreads();
	}
}

// log det(1 + U D V) = sum log D_b + sum log|R_ii| of X = Q R; the sign from the R_ii, det Q and
// det U (-1 per reflector: nref[1], nref[0]).  A zero R_ii: log|det| = -inf, recorded as singular.
__global__ __launch_bounds__(256) void stab_logdet_kernel(const double *__restrict__ d, const double *__restrict__ zr,
		unsigned n, const int *__restrict__ nref, double *__restrict__ scal)
{
	__shared__ double part[256];
	__shared__ int negs[256], sing[256];
	const int tid = threadIdx.x;
	double s = 0;
	int neg = 0, sg = 0;
	for(unsigned i = tid; i < n; i += 256){
		const double r = zr[(size_t)i * n + i];
		s += (d[i] > 1 ? log(d[i]) : 0.0) + log(fabs(r));
		neg += r < 0;
		if(r == 0) sg = max(sg, (int)i + 1);
	}
	part[tid] = s;
	negs[tid] = neg;
	sing[tid] = sg;
	__syncthreads();
	for(int off = 128; off > 0; off >>= 1){
		if(tid < off){
			part[tid] += part[tid + off];
			negs[tid] += negs[tid + off];
			sing[tid] = max(sing[tid], sing[tid + off]);
		}
		__syncthreads();
	}
	if(tid == 0){
		scal[SCAL_LOGDET] = sing[0] ? -HUGE_VAL : part[0];
		scal[SCAL_SIGN] = (!sing[0] && ((negs[0] + nref[0] + nref[1]) & 1)) ? -1.0 : 1.0;
		scal[SCAL_SINGULAR] = sing[0];
		scal[SCAL_SCHUR_FAIL] = 0;
	}
}


// Panel width: 32 columns, or 16 above 1024 sites, where 512 threads still hold a panel (16 rows of 4 columns each).
static unsigned qr_nb(unsigned n){ return n <= 1024 ? 32u : 16u; }

// Leading dimension of the reflectors: 64-row blocks from any panel's first row stay inside a column.
static unsigned qr_ldv(unsigned n){ return (n + 63) / 64 * 64 + 64; }

// buffers of the stabilised product, allocated together on first use (or at creation when
// ephmc_config.stabilize is set)
int stab_reserve(ephmc_ctx *c)
{
	if(c->stab.U) return EPHMC_OK;
	const size_t mat = c->mat, n = c->ns, nb = qr_nb(c->ns), tsz = (n + nb - 1) / nb * nb * nb;
	double **d[] = {&c->stab.U, &c->stab.V[0], &c->stab.V[1], &c->stab.ZR, &c->stab.d, &c->stab.key, &c->stab.T, &c->stab.Rinv, &c->stab.Vm};
	const size_t vsz = (n + nb - 1) / nb * nb * qr_ldv(c->ns), sz[] = {mat, mat, mat, mat, n, n, tsz, tsz, vsz};
	for(int i = 0; i < 9; i++){
		if(hipMalloc((void **)d[i], sz[i] * sizeof(double)) != hipSuccess){
			(void)hipGetLastError();
			stab_release(c);
			set_error("stabilised product: device buffers (%zu MB) could not be allocated", (5 * mat * 8) >> 20);
			return EPHMC_ERR_ALLOC;
		}
	}
	if(hipMalloc((void **)&c->stab.perm, n * sizeof(int)) != hipSuccess
		|| hipMalloc((void **)&c->stab.nref, 2 * sizeof(int)) != hipSuccess){
		(void)hipGetLastError();
		stab_release(c);
		set_error("stabilised product: device buffers could not be allocated");
		return EPHMC_ERR_ALLOC;
	}
	return EPHMC_OK;
}

void stab_release(ephmc_ctx *c)
{
	void *b[] = {c->stab.U, c->stab.V[0], c->stab.V[1], c->stab.ZR, c->stab.d, c->stab.key, c->stab.T, c->stab.Rinv, c->stab.Vm,
		c->stab.perm, c->stab.nref};
	for(void *p : b) if(p) (void)hipFree(p);
	c->stab = StabWork{};
}

// Start of a product: d = 1, and the reflectors 0 (the factorisations write only their support).  On the
// context's stream in every call, so that the products are ordered behind it, captured or not, and its
// launch is the one that d needs anyway (0.65 MB of reflectors at N = 256, 34 MB at 2025).
__global__ __launch_bounds__(256) void stab_start_kernel(double *__restrict__ d, unsigned n, double *__restrict__ vm, size_t vsz)
{
	const size_t t = blockIdx.x * (size_t)256 + threadIdx.x;
	if(t < n) d[t] = 1.0;
	for(size_t e = t; e < vsz; e += (size_t)gridDim.x * 256) vm[e] = 0.0;
}

// Blocked QR of z in place: T factors to w.T, number of nonzero reflectors to nref.  Each launch's
// workgroup shape is the smallest whose registers hold the rows of the panel it factorises.
static int blocked_qr(ephmc_ctx *c, double *z, int *nref)
{
	const unsigned n = c->ns, nb = qr_nb(n), np = (n + nb - 1) / nb;
	double *tm = c->stab.T, *vm = c->stab.Vm;
	const unsigned ldv = qr_ldv(n);
	for(int p = -1; p + 1 < (int)np; p++){
		const unsigned j1 = (unsigned)(p + 1) * nb, m = n - j1;
		const unsigned grid = 1 + (p >= 0 && n > j1 + nb ? (n - j1 - nb + 15) / 16 : 0);
		if(nb == 16) qr_step_kernel<16, 512, 16><<<grid, 512, 0, c->stream>>>(z, n, p, vm, ldv, tm, nref);
		else if(m <= 128) qr_step_kernel<32, 256, 4><<<grid, 256, 0, c->stream>>>(z, n, p, vm, ldv, tm, nref);
		else if(m <= 256) qr_step_kernel<32, 256, 8><<<grid, 256, 0, c->stream>>>(z, n, p, vm, ldv, tm, nref);
		else if(m <= 512) qr_step_kernel<32, 512, 8><<<grid, 512, 0, c->stream>>>(z, n, p, vm, ldv, tm, nref);
		else qr_step_kernel<32, 512, 16><<<grid, 512, 0, c->stream>>>(z, n, p, vm, ldv, tm, nref);
		EPHMC_LAUNCHED();
	}
	return EPHMC_OK;
}

// minv = (1 + B_0 ... B_{nt-1})^{-1} and its log det (scal[SCAL_LOGDET], sign in SCAL_SIGN) with the
// slice products in precision prec and an FP64 QR every k slices; the coefficients of the field
// must be current for prec.  Scratch: the buffers above, d_Tfin / d_Tfin32 (block products).
int stable_logdet_inverse(ephmc_ctx *c, int prec, unsigned k, double *minv)
{
	const unsigned n = c->ns, nt = c->nt;
	if(n > 2048){ set_error("stabilised product: N = %u exceeds 2048", n); return EPHMC_ERR_UNSUPPORTED; }
	if(k == 0) k = 1;
	EPHMC_TRY(stab_reserve(c));
	StabWork &w = c->stab;
	EPHMC_TRY(set_identity(c, EPHMC_FP64, w.U));
	EPHMC_TRY(set_identity(c, EPHMC_FP64, w.V[0]));
	void *Y = prec == EPHMC_FP64 ? (void *)c->d_Tfin : (void *)c->d_Tfin32;
	const unsigned nb = qr_nb(n), np = (n + nb - 1) / nb, tiles = (n + 15) / 16, ldv = qr_ldv(n);
	const size_t vsz = (size_t)np * nb * ldv;
	stab_start_kernel<<<(unsigned)std::min<size_t>((vsz + 255) / 256, 2048), 256, 0, c->stream>>>(w.d, n, w.Vm, vsz);
	EPHMC_LAUNCHED();
	const dim3 tg((n + 31) / 32, (n + 31) / 32);
	int cur = 0;
	for(int hi = (int)nt - 1; hi >= 0; hi -= (int)k){
		const int cnt = std::min<int>((int)k, hi + 1);
		// Y = B_{hi-cnt+1} ... B_hi U: slices hi down to hi-cnt+1, each applied from the left
		EPHMC_TRY(chain_range(c, prec, w.U, Y, hi, -1, cnt));
		if(prec == EPHMC_FP64){
			qr_key_kernel<double><<<(n + 3) / 4, 256, 0, c->stream>>>((const double *)Y, w.d, n, w.key);
			qr_sort_kernel<double><<<n, 256, 0, c->stream>>>((const double *)Y, w.d, w.key, n, w.ZR, w.perm);
		}else{
			qr_key_kernel<float><<<(n + 3) / 4, 256, 0, c->stream>>>((const float *)Y, w.d, n, w.key);
			qr_sort_kernel<float><<<n, 256, 0, c->stream>>>((const float *)Y, w.d, w.key, n, w.ZR, w.perm);
		}
		EPHMC_LAUNCHED();
		EPHMC_TRY(blocked_qr(c, w.ZR, w.nref));
		if(nb == 32) qr_form_q_kernel<32><<<tiles, 256, 0, c->stream>>>(w.Vm, ldv, w.T, n, w.U);
		else qr_form_q_kernel<16><<<tiles, 256, 0, c->stream>>>(w.Vm, ldv, w.T, n, w.U);
		EPHMC_LAUNCHED();
		qr_update_v_kernel<<<tg, 256, n * sizeof(int), c->stream>>>(w.ZR, w.perm, n, w.V[cur], w.V[cur ^ 1], w.d);
		EPHMC_LAUNCHED();
		cur ^= 1;
	}
	stab_x_kernel<<<tg, 256, 0, c->stream>>>(w.U, w.V[cur], w.d, n, w.ZR);
	EPHMC_LAUNCHED();
	EPHMC_TRY(blocked_qr(c, w.ZR, w.nref + 1));
	if(nb == 32){
		tri_inverse_kernel<32><<<np, 256, 0, c->stream>>>(w.ZR, n, w.Rinv);
		stab_solve_kernel<32><<<tiles, 256, 0, c->stream>>>(w.ZR, w.Vm, ldv, w.T, w.Rinv, w.U, w.d, n, minv);
	}else{
		tri_inverse_kernel<16><<<np, 256, 0, c->stream>>>(w.ZR, n, w.Rinv);
		stab_solve_kernel<16><<<tiles, 256, 0, c->stream>>>(w.ZR, w.Vm, ldv, w.T, w.Rinv, w.U, w.d, n, minv);
	}
	EPHMC_LAUNCHED();
	stab_logdet_kernel<<<1, 256, 0, c->stream>>>(w.d, w.ZR, n, w.nref, c->d_scal);
	EPHMC_LAUNCHED();
	return EPHMC_OK;
}

} // namespace ephmc

using namespace ephmc;

extern "C" int ephmc_stable_logdet_inv(ephmc_ctx *c, const double *x, int precision, unsigned k, double *M_inv,
		double *logdet, int *sign)
{
	if(!c || !x || !M_inv){ set_error("null argument"); return EPHMC_ERR_ARG; }
	if(precision != EPHMC_FP64 && precision != EPHMC_MIXED){ set_error("precision"); return EPHMC_ERR_ARG; }
	if(c->cfg.zero_filling || c->cfg.single_particle){
		set_error("the stabilised product forms 1 + B..B: not for ZERO_FILLING / SINGLE_PARTICLE");
		return EPHMC_ERR_UNSUPPORTED;
	}
	if(precision == EPHMC_MIXED && !c->d_coef32){
		set_error("FP32 slices need a context created with EPHMC_MIXED");
		return EPHMC_ERR_ARG;
	}
	EPHMC_TRY(coefficients(c, x, precision == EPHMC_MIXED));
	EPHMC_TRY(stable_logdet_inverse(c, precision, k, M_inv));
	if(!logdet && !sign) return EPHMC_OK;
	double s[SCAL_COUNT];
	EPHMC_HIP(hipMemcpyAsync(s, c->d_scal, sizeof(s), hipMemcpyDeviceToHost, c->stream));
	EPHMC_HIP(hipStreamSynchronize(c->stream));
	if(logdet) *logdet = s[SCAL_LOGDET];
	if(sign) *sign = s[SCAL_SIGN] < 0 ? -1 : 1;
	if(s[SCAL_SINGULAR] != 0 || s[SCAL_LOGDET] == -HUGE_VAL){
		set_error("singular matrix in the stabilised inverse; log|det| = -inf");
		return EPHMC_ERR_NUMERIC;
	}
	return EPHMC_OK;
}
